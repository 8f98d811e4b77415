// ocfd_mlp_net.h -- loss and gradients of a network whose padded widths are
// all at most 256, in three launches.  Included by ocfd_mlp.hip.
//
// As one GEMM per layer and direction a batch of 8192 was 36 launches in a
// chain, 4 to 18 us each, of matrix products that take 1 us at the card's
// rate: bound by launches, by column sums and by transposing both operands of
// dW through LDS.  A sample's forward and backward passes touch no other
// sample, so:
//   k_net      a workgroup carries 32 samples through every layer, the loss
//              and back, activations in LDS; it leaves each layer's input and
//              dZ as MFMA operands for the sum over samples (32 samples are
//              one K chunk), and its share of the bias gradients;
//   k_net_dw   dW of all layers, 64 x 64 tiles by K splits, operands straight
//              from memory into registers;
//   k_net_sum  adds the splits and shares in a fixed order into the gradient
//              arrays and the flat layout.
// 12-256x5-9, batch 8192: 464 us a call as GEMMs, 61 so (k_net 41, k_net_dw
// 16, k_net_sum 6 under the profiler).  A sample's values are those of the GEMM
// path bit for bit (same K order); sums over samples, and the loss's over the
// outputs, differ in order.
#pragma once

constexpr int NET_R = 32, NET_NW = 8, NET_W = 256, NET_LD = NET_W + 8, NET_S = 8;

// Position of W[o][k] in MFMA operand order over k: for the forward pass of
// W [doutp][dinp]; with the arguments exchanged that of the transpose.
__host__ __device__ inline long net_frag(int o, int k, int kp) {
  return ((long)((o >> 4) * (kp >> 5) + (k >> 5)) * 64 + ((k >> 3) & 3) * 16 + (o & 15)) * 8 + (k & 7);
}

struct NetLayer {
  int din, dout, dinp, doutp;
  const bf16 *Wf, *Wt;  // W and its transpose in operand order
  const float* b;
  bf16 *At, *Dt;        // the layer's input and dZ, operands of dW: [width/16][chunk][64 lanes][8]
  float* gp;            // GELU'(Z) of a hidden layer, in accumulator order
  float* cs;            // [chunk][doutp] shares of the bias gradient
  float *gW, *gb;
  long flat;            // the layer's offset in the flat gradient
  int tile0;            // first 64 x 64 tile of dW
};
struct NetArgs {
  int L, nblk, tiles, bias_blocks;
  long B;
  const float *x, *y;
  double* lp;   // [chunk] sums of squared errors
  float* part;  // [tile][NET_S][4096] K splits of dW
  float *grad, *loss, *loss2;
  NetLayer l[MLP_MAX_LAYERS];
};

// acc[j][i] = rows 16 i .. of H [32][32 KS] times columns 16 (w + 8 j) .. of
// the operand at Wp, NJ column tiles a wave of nt in all (a wave beyond them
// repeats the last, to no effect).  The weights do not wait for the
// activations: their loads (all K chunks) are issued ahead of the barrier.
template <int KS, int NJ>
__device__ __forceinline__ void net_mm(const bf16 (*H)[NET_LD], const bf16* __restrict__ Wp, int nt, int w, int lane,
                                       floatx4 (*acc)[2]) {
  bf16x8 wf[NJ][KS];
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const long jb = min(w + NET_NW * j, nt - 1);
#pragma unroll
    for (int s = 0; s < KS; s++) wf[j][s] = *(const bf16x8*)&Wp[((jb * KS + s) * 64 + lane) * 8];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NJ; j++)
#pragma unroll
    for (int i = 0; i < 2; i++) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < KS; s++) {
    bf16x8 a[2];
#pragma unroll
    for (int i = 0; i < 2; i++) a[i] = *(const bf16x8*)&H[16 * i + (lane & 15)][32 * s + (lane >> 4) * 8];
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int i = 0; i < 2; i++)
        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], wf[j][s], acc[j][i], 0, 0, 0);
  }
}
template <int KS>
__device__ __forceinline__ void net_mm_n(const bf16 (*H)[NET_LD], const bf16* __restrict__ Wp, int nt, int w, int lane,
                                         floatx4 (*acc)[2]) {
  if (nt > NET_NW) net_mm<KS, 2>(H, Wp, nt, w, lane, acc);
  else net_mm<KS, 1>(H, Wp, nt, w, lane, acc);
}
// K and N padded widths (multiples of 64, at most 256); returns the wave's
// number of column tiles
__device__ __forceinline__ int net_product(const bf16 (*H)[NET_LD], const bf16* __restrict__ Wp, int K, int N, int w,
                                           int lane, floatx4 (*acc)[2]) {
  const int nt = N >> 4;
  switch (K >> 6) {
    case 1: net_mm_n<2>(H, Wp, nt, w, lane, acc); break;
    case 2: net_mm_n<4>(H, Wp, nt, w, lane, acc); break;
    case 3: net_mm_n<6>(H, Wp, nt, w, lane, acc); break;
    default: net_mm_n<8>(H, Wp, nt, w, lane, acc); break;
  }
  return (w < nt) + (w + NET_NW < nt);
}

// An accumulator tile (column 16 jb + lane % 16, rows 16 i + 4 (lane / 16) +
// r) as bf16 into the rows of H and into the operand for the sum over rows.
__device__ __forceinline__ void net_put(bf16 (*H)[NET_LD], bf16* __restrict__ T, long nblk, long blk, int jb, int i,
                                        int lane, floatx4 v) {
  const int lr = lane & 15, lg = lane >> 4;
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
  bf16x4 h;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    h[r] = (bf16)v[r];
    H[16 * i + 4 * lg + r][16 * jb + lr] = h[r];
  }
  *(bf16x4*)&T[(jb * nblk + blk) * 512 + (16 * (2 * i + (lg >> 1)) + lr) * 8 + 4 * (lg & 1)] = h;
}

// The tile pair's column sums over the 32 rows
__device__ __forceinline__ void net_colsum(float* __restrict__ cs, int jb, int lane, const floatx4* v) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int r = 0; r < 4; r++) s += v[i][r];
  s += __shfl_xor(s, 16, 64);
  s += __shfl_xor(s, 32, 64);
  if (lane < 16) cs[16 * jb + lane] = s;
}

// Bound by latency along the chain of layers (each: weights from L2, a
// barrier, 8 LDS reads and 32 MFMAs a wave, the GELU): 32 rows give a batch
// of 8192 a workgroup on every CU.
__global__ __launch_bounds__(64 * NET_NW) void k_net(NetArgs P) {
  __shared__ __attribute__((aligned(16))) bf16 H[2][NET_R][NET_LD];
  __shared__ double sl[NET_NW];
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const long blk = blockIdx.x, nblk = P.nblk, r0 = blk * NET_R;
  {
    const int din = P.l[0].din, dinp = P.l[0].dinp;
    for (int e = t; e < NET_R * dinp; e += 64 * NET_NW) {
      const int r = e / dinp, c = e % dinp;
      H[0][r][c] = (bf16)((r0 + r < P.B && c < din) ? P.x[(r0 + r) * din + c] : 0.f);
    }
    __syncthreads();
    for (int e = t; e < dinp * 4; e += 64 * NET_NW) {
      const int ct = e >> 6, fl = e & 63;
      bf16x8 v;
#pragma unroll
      for (int q = 0; q < 8; q++) v[q] = H[0][8 * (fl >> 4) + q][16 * ct + (fl & 15)];
      *(bf16x8*)&P.l[0].At[(ct * nblk + blk) * 512 + fl * 8] = v;
    }
  }
  int cur = 0;
  floatx4 acc[2][2];
  for (int l = 0; l < P.L - 1; l++, cur ^= 1) {
    const NetLayer& y = P.l[l];
    const int nj = net_product(H[cur], y.Wf, y.dinp, y.doutp, w, lane, acc);
    for (int j = 0; j < nj; j++) {
      const int jb = w + NET_NW * j;
      const float bias = y.b[16 * jb + lr];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        floatx4 h, g;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float z = (j ? acc[1][i][r] : acc[0][i][r]) + bias;
          h[r] = gelu_f(z);
          g[r] = dgelu_f(z);
        }
        net_put(H[cur ^ 1], P.l[l + 1].At, nblk, blk, jb, i, lane, h);
        *(floatx4*)&y.gp[(((blk * (y.doutp >> 4) + jb) * 2 + i) * 64 + lane) * 4] = g;
      }
    }
  }
  double e2 = 0.0;  // a lane adds up to 16 squares of one column: as floats they may overflow together
  {
    const NetLayer& y = P.l[P.L - 1];
    const int nj = net_product(H[cur], y.Wf, y.dinp, y.doutp, w, lane, acc);
    const float cnt = (float)(P.B * y.dout);
    for (int j = 0; j < nj; j++) {
      const int jb = w + NET_NW * j, c = 16 * jb + lr;
      const float bias = y.b[c];
      floatx4 g[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const long row = r0 + 16 * i + 4 * lg + r;
          g[i][r] = 0.f;
          if (row < P.B && c < y.dout) {
            const float e = ((j ? acc[1][i][r] : acc[0][i][r]) + bias) - P.y[row * y.dout + c];
            e2 += (double)e * (double)e;
            g[i][r] = 2.0f * e / cnt;
          }
        }
        net_put(H[cur ^ 1], y.Dt, nblk, blk, jb, i, lane, g[i]);
      }
      net_colsum(y.cs + blk * y.doutp, jb, lane, g);
    }
    cur ^= 1;
  }
  for (int o = 32; o > 0; o >>= 1) e2 += __shfl_xor(e2, o, 64);
  if (lane == 0) sl[w] = e2;
  __syncthreads();
  if (t == 0) {
    double s = 0.0;
    for (int k = 0; k < NET_NW; k++) s += sl[k];
    P.lp[blk] = s;
  }
  for (int l = P.L - 1; l > 0; l--, cur ^= 1) {
    const NetLayer& y = P.l[l];
    const NetLayer& p = P.l[l - 1];
    const int nj = net_product(H[cur], y.Wt, y.doutp, y.dinp, w, lane, acc);
    for (int j = 0; j < nj; j++) {
      const int jb = w + NET_NW * j;
      floatx4 v[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const floatx4 g = *(const floatx4*)&p.gp[(((blk * (p.doutp >> 4) + jb) * 2 + i) * 64 + lane) * 4];
#pragma unroll
        for (int r = 0; r < 4; r++) v[i][r] = (j ? acc[1][i][r] : acc[0][i][r]) * g[r];
        net_put(H[cur ^ 1], p.Dt, nblk, blk, jb, i, lane, v[i]);
      }
      net_colsum(p.cs + blk * p.doutp, jb, lane, v);
    }
  }
}

// dW[m][n] = sum over samples of dZ[.][m] A[.][n]: workgroup (split, tile),
// the split running over the XCDs: chunk c was written by the XCD c % 8, whose
// L2 the split c % 8 reads.  The four waves take every fourth chunk of the
// split and meet in LDS.
__global__ __launch_bounds__(256) void k_net_dw(NetArgs P) {
  __shared__ __attribute__((aligned(16))) float red[4][4096];
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int split = blockIdx.x, tile = blockIdx.y;
  int l = 0;
  while (l + 1 < P.L && tile >= P.l[l + 1].tile0) l++;
  const NetLayer& y = P.l[l];
  const int nt = y.dinp >> 6, tm = (tile - y.tile0) / nt, tn = (tile - y.tile0) % nt;
  const long nblk = P.nblk;
  const bf16* __restrict__ D = y.Dt + 4 * tm * nblk * 512 + lane * 8;
  const bf16* __restrict__ A = y.At + 4 * tn * nblk * 512 + lane * 8;
  floatx4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  bf16x8 a[4], b[4];
  long c = split + NET_S * w;
  if (c < nblk) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      a[i] = *(const bf16x8*)&D[(i * nblk + c) * 512];
      b[i] = *(const bf16x8*)&A[(i * nblk + c) * 512];
    }
  }
  while (c < nblk) {
    const long cn = c + 4 * NET_S;
    bf16x8 an[4], bn[4];
    if (cn < nblk) {  // the next chunk's operands, in flight during the products
#pragma unroll
      for (int i = 0; i < 4; i++) {
        an[i] = *(const bf16x8*)&D[(i * nblk + cn) * 512];
        bn[i] = *(const bf16x8*)&A[(i * nblk + cn) * 512];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      a[i] = an[i];
      b[i] = bn[i];
    }
    c = cn;
  }
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) *(floatx4*)&red[w][((4 * i + j) * 64 + lane) * 4] = acc[i][j];
  __syncthreads();
  float* __restrict__ out = P.part + ((long)tile * NET_S + split) * 4096;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int e = (k * 256 + t) * 4;
    const floatx4 s = ((*(const floatx4*)&red[0][e] + *(const floatx4*)&red[1][e]) + *(const floatx4*)&red[2][e]) +
                      *(const floatx4*)&red[3][e];
    *(floatx4*)&out[e] = s;
  }
}

// Splits and shares added in a fixed order: four blocks a tile of dW, one per
// 64 biases, one for the loss.
__global__ __launch_bounds__(256) void k_net_sum(NetArgs P) {
  const int t = threadIdx.x;
  int b = blockIdx.x;
  if (b < 4 * P.tiles) {
    const int tile = b >> 2, e = (b & 3) * 256 + t;  // four rows of a column
    int l = 0;
    while (l + 1 < P.L && tile >= P.l[l + 1].tile0) l++;
    const NetLayer& y = P.l[l];
    const int nt = y.dinp >> 6, tm = (tile - y.tile0) / nt, tn = (tile - y.tile0) % nt;
    const float* __restrict__ in = P.part + (long)tile * NET_S * 4096 + e * 4;
    floatx4 v[NET_S], s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NET_S; k++) v[k] = *(const floatx4*)&in[k * 4096];
#pragma unroll
    for (int k = 0; k < NET_S; k++) s += v[k];
    const int lane = e & 63, i = e >> 8, j = (e >> 6) & 3;
    const int m = 64 * tm + 16 * i + 4 * (lane >> 4), n = 64 * tn + 16 * j + (lane & 15);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      y.gW[(long)(m + r) * y.dinp + n] = s[r];
      if (P.grad && m + r < y.dout && n < y.din) P.grad[y.flat + (long)(m + r) * y.din + n] = s[r];
    }
    return;
  }
  b -= 4 * P.tiles;
  if (b < P.bias_blocks) {
    __shared__ float red[4][64];
    int l = 0;
    while (b >= P.l[l].doutp >> 6) b -= P.l[l++].doutp >> 6;
    const NetLayer& y = P.l[l];
    const int c = 64 * b + (t & 63), q = t >> 6;
    float s = 0.f;
#pragma unroll 8
    for (int k = q; k < P.nblk; k += 4) s += y.cs[(long)k * y.doutp + c];
    red[q][t & 63] = s;
    __syncthreads();
    if (q == 0) {
      const float v = (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
      y.gb[c] = v;
      if (P.grad && c < y.dout) P.grad[y.flat + (long)y.dout * y.din + c] = v;
    }
    return;
  }
  __shared__ double rd[256];
  double s = 0.0;
  for (int k = t; k < P.nblk; k += 256) s += P.lp[k];
  rd[t] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h) rd[t] += rd[t + h];
    __syncthreads();
  }
  if (t == 0) {
    const float v = (float)(rd[0] / (double)(P.B * P.l[P.L - 1].dout));
    P.loss[0] = v;
    if (P.loss2) P.loss2[0] = v;
  }
}
