// Fused passes of the learned warm start's network (included by mlp.hip).
//
// k_net runs the whole network for 16 rows per workgroup: inputs built from
// the caller's rows (normalised, or gathered from the training set), three
// layers, and in training the loss gradient and both backward layers, with
// every activation in LDS or registers. k_wgrad then forms all weight and bias
// gradients and applies AdamW: two launches per training batch.
//
// What bounds them: latency. A 4096 x 195-256-256-18 batch is 2.5 GFLOP (2 us
// at the card's measured 1.2 PFLOP/s) and 10 MB of activations (2 us); a
// workgroup's chain of five dependent products, each waiting for its weights
// from L2, and k_wgrad's first touch of what other XCDs wrote take the time. Hence 16
// rows per workgroup (256 workgroups for a batch of 4096: one per CU), weights
// loaded straight into MFMA fragments (no LDS staging: no wave shares a
// fragment with another) a few K steps ahead, the next layer's first
// fragments before the barrier that ends the previous one, and activations
// stored transposed ([column][row]), which makes k_wgrad's operands
// contiguous along its K = row dimension.
//
// Measured (MI355X, 195-256-256-18): a training batch of 4096 rows 183 us in 23
// launches -> 51 us in two (k_net 29.5, k_wgrad 21.7); inference of 2000 envs
// (features packed, three products) 38 -> 17.5 us; one epoch over 131072 rows
// with the host's shuffle 6.09 -> 2.04 ms; a gradient call on 4096 host rows
// 555 -> 240 us (the rows now go to the device as they are).
//
// The arithmetic is that of the separate kernels below (same MFMA K order,
// same split-K and column-sum slices, added in the same order), so results are
// the same bits. Widths beyond net_fused()'s limits take the separate kernels.
#pragma once

enum { FROWS = 16, FWAVES = 8, FTHREADS = 64 * FWAVES };

struct NetView {
  int nin, ip, nh, op, nout;
  const uint16_t *W1t, *W2t, *W3t;  // bf16 weights transposed: [outputs][inputs], forward products
  const uint16_t *W2, *W3;          // bf16 weights [inputs][outputs], backward products
  const float *b1, *b2, *b3;
};

// network inputs: row r is raw[idx ? idx[r] : r][0 .. nin), columns [coff,
// coff + nu) taken from ctrl[r] (zeros when null), normalised by mean / istd
// when set; rows at or beyond nrow are zero
struct XSrc {
  const float* raw;
  const int* idx;
  const float* ctrl;
  int coff, nu, nrow;
  const float *mean, *istd;
};

// inference outputs y[r][0 .. ny): (network * oscale + oshift when set) + base when set
struct NetOut {
  float* y;
  int ny;
  const float *oscale, *oshift, *base;
  int ldbase;
};

// training: targets tgt[idx ? idx[r] : r][0 .. nout), standardised by omean /
// ostd when set, of the first rvalid rows; rp rows in all (a multiple of 32).
// Activations and gradients as bf16 [column][rp], gradients also as fp32
// [column][rp] (bias sums); per-row loss.
struct NetTrain {
  const float *tgt, *omean, *ostd;
  int rvalid, rp;
  float scale;
  uint16_t *xt, *h1t, *h2t, *d1t, *d2t, *d3t;
  float *f1, *f2, *f3, *rowloss;
};

// fragments of PF K steps (32 wide) x NT column tiles (16 wide) of a weight
// matrix stored [column][K]: lane l holds column l % 16, K entries 8 (l / 16) ..
template <int NT, int PF>
__device__ __forceinline__ void net_load(v8bf (&b)[PF][NT], const uint16_t* __restrict__ W, int K, int ntile, int wave,
                                         int lane, int kt0) {
#pragma unroll
  for (int p = 0; p < PF; p++)
#pragma unroll
    for (int t = 0; t < NT; t++) {
      int ct = wave + FWAVES * t;
      if (32 * (kt0 + p) < K && ct < ntile)
        b[p][t] = *reinterpret_cast<const v8bf*>(W + (size_t)(16 * ct + (lane & 15)) * K + 32 * (kt0 + p) + 8 * (lane >> 4));
    }
}

template <int NT, int PF>
__device__ __forceinline__ void net_mfma(v4f (&acc)[NT], const v8bf (&b)[PF][NT], const uint16_t* A, int lda, int K,
                                         int ntile, int wave, int lane, int kt0) {
#pragma unroll
  for (int p = 0; p < PF; p++) {
    if (32 * (kt0 + p) >= K) continue;
    v8bf a = *reinterpret_cast<const v8bf*>(A + (lane & 15) * lda + 32 * (kt0 + p) + 8 * (lane >> 4));
#pragma unroll
    for (int t = 0; t < NT; t++)
      if (wave + FWAVES * t < ntile) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[p][t], acc[t], 0, 0, 0);
  }
}

// acc[t] = A[16][K] (LDS) times column tile wave + 8 t of W; b0 holds the first PF K steps
template <int NT, int PF>
__device__ __forceinline__ void net_mm(v4f (&acc)[NT], v8bf (&b0)[PF][NT], const uint16_t* A, int lda,
                                       const uint16_t* __restrict__ W, int K, int ntile, int wave, int lane) {
  v8bf b1[PF][NT] = {};
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  for (int kt = 0; 32 * kt < K; kt += 2 * PF) {
    net_load<NT, PF>(b1, W, K, ntile, wave, lane, kt + PF);
    net_mfma<NT, PF>(acc, b0, A, lda, K, ntile, wave, lane, kt);
    net_load<NT, PF>(b0, W, K, ntile, wave, lane, kt + 2 * PF);
    net_mfma<NT, PF>(acc, b1, A, lda, K, ntile, wave, lane, kt + PF);
  }
}

__device__ __forceinline__ void store4(uint16_t* p, const uint16_t* v) {
  *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)v[0] | ((uint32_t)v[1] << 16), (uint32_t)v[2] | ((uint32_t)v[3] << 16));
}

size_t net_lds(int ip, int nh, int op) {
  return (size_t)FROWS * 2 * ((ip + 8) + 2 * (nh + 8) + (op + 8)) + (size_t)FROWS * 4 * op;
}

// hidden-layer epilogue: z = acc + bias kept in zk, silu(z) as bf16 to LDS
// [row][column] and, in training, to ht [column][rp]
template <int NT, bool TRAIN>
__device__ __forceinline__ void net_hidden(const v4f (&acc)[NT], float (&zk)[NT][4], const float* __restrict__ bias,
                                           int ntile, int wave, int lane, uint16_t* H, int ldh, uint16_t* ht, int rp,
                                           int r0) {
#pragma unroll
  for (int t = 0; t < NT; t++) {
    int ct = wave + FWAVES * t;
    if (ct >= ntile) continue;
    int c = 16 * ct + (lane & 15), r = 4 * (lane >> 4);
    float bb = bias[c];
    uint16_t hv[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float z = acc[t][i] + bb;
      zk[t][i] = z;
      hv[i] = f2bf(silu(z));
      H[(r + i) * ldh + c] = hv[i];
    }
    if (TRAIN) store4(ht + (size_t)c * rp + r0 + r, hv);
  }
}

// backward epilogue: g = dY silu'(z); bf16 to LDS (when H) and dt, fp32 to f
template <int NT>
__device__ __forceinline__ void net_back(const v4f (&acc)[NT], const float (&zk)[NT][4], int ntile, int wave, int lane,
                                         uint16_t* H, int ldh, uint16_t* dt, float* f, int rp, int r0) {
#pragma unroll
  for (int t = 0; t < NT; t++) {
    int ct = wave + FWAVES * t;
    if (ct >= ntile) continue;
    int c = 16 * ct + (lane & 15), r = 4 * (lane >> 4);
    uint16_t dv[4];
    float gv[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float z = zk[t][i];
      gv[i] = silu_bwd(acc[t][i], z);
      dv[i] = f2bf(gv[i]);
      if (H) H[(r + i) * ldh + c] = dv[i];
    }
    store4(dt + (size_t)c * rp + r0 + r, dv);
    *reinterpret_cast<float4*>(f + (size_t)c * rp + r0 + r) = make_float4(gv[0], gv[1], gv[2], gv[3]);
  }
}

// NT: column tiles of a hidden layer per wave (nh <= 128 NT)
template <int NT, bool TRAIN>
__global__ void __launch_bounds__(FTHREADS) k_net(NetView n, XSrc x, NetOut o, NetTrain tr) {
  constexpr int PF = 8 / NT;
  extern __shared__ __align__(16) uint16_t net_sm[];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r0 = blockIdx.x * FROWS;
  const int lx = n.ip + 8, lh = n.nh + 8, l3 = n.op + 8, ht = n.nh / 16, ot = n.op / 16;
  uint16_t *X = net_sm, *H1 = X + FROWS * lx, *H2 = H1 + FROWS * lh, *D3 = H2 + FROWS * lh;
  float* O = reinterpret_cast<float*>(D3 + FROWS * l3);
  v8bf b[PF][NT] = {};
  v4f acc[NT];
  float z1[NT][4], z2[NT][4];
  net_load<NT, PF>(b, n.W1t, n.ip, ht, wave, lane, 0);
  // inputs: two rows per wave
  for (int rr = wave; rr < FROWS; rr += FWAVES) {
    int r = r0 + rr;
    bool in = r < x.nrow;
    const float* src = x.raw + (size_t)(in ? (x.idx ? x.idx[r] : r) : 0) * n.nin;
    for (int c = lane; c < n.ip; c += 64) {
      float v = 0.f;
      if (in && c < n.nin) {
        if (c >= x.coff && c < x.coff + x.nu) v = x.ctrl ? x.ctrl[(size_t)r * x.nu + c - x.coff] : 0.f;
        else v = src[c];
        if (x.mean) v = (v - x.mean[c]) * x.istd[c];
      }
      X[rr * lx + c] = f2bf(v);
    }
  }
  __syncthreads();
  if (TRAIN)
    for (int c = tid; c < n.ip; c += FTHREADS) {
      v8u a[2];
#pragma unroll
      for (int i = 0; i < FROWS; i++) a[i >> 3][i & 7] = X[i * lx + c];
      v8u* dst = reinterpret_cast<v8u*>(tr.xt + (size_t)c * tr.rp + r0);
      dst[0] = a[0];
      dst[1] = a[1];
    }
  net_mm<NT, PF>(acc, b, X, lx, n.W1t, n.ip, ht, wave, lane);
  net_load<NT, PF>(b, n.W2t, n.nh, ht, wave, lane, 0);
  net_hidden<NT, TRAIN>(acc, z1, n.b1, ht, wave, lane, H1, lh, tr.h1t, tr.rp, r0);
  __syncthreads();
  net_mm<NT, PF>(acc, b, H1, lh, n.W2t, n.nh, ht, wave, lane);
  v8bf bo[8][1] = {};
  v4f ao[1];
  net_load<1, 8>(bo, n.W3t, n.nh, ot, wave, lane, 0);
  net_hidden<NT, TRAIN>(acc, z2, n.b2, ht, wave, lane, H2, lh, tr.h2t, tr.rp, r0);
  __syncthreads();
  net_mm<1, 8>(ao, bo, H2, lh, n.W3t, n.nh, ot, wave, lane);
  if (wave < ot) {
    int c = 16 * wave + (lane & 15);
    float bb = n.b3[c];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      int rr = 4 * (lane >> 4) + i;
      float y = ao[0][i] + bb;
      if (TRAIN) {
        O[rr * n.op + c] = y;
      } else if (c < o.ny && r0 + rr < x.nrow) {
        float yo = o.oscale ? y * o.oscale[c] + o.oshift[c] : y;
        if (o.base) yo += o.base[(size_t)(r0 + rr) * o.ldbase + c];
        o.y[(size_t)(r0 + rr) * o.ny + c] = yo;
      }
    }
  }
  if (!TRAIN) return;
  net_load<NT, PF>(b, n.W3, n.op, ht, wave, lane, 0);
  __syncthreads();
  for (int t = tid; t < FROWS * n.op; t += FTHREADS) {
    int rr = t & (FROWS - 1), c = t / FROWS, r = r0 + rr;
    float g = 0.f, d = 0.f;
    if (r < tr.rvalid && c < n.nout) {
      float y = tr.tgt[(size_t)(x.idx ? x.idx[r] : r) * n.nout + c];
      if (tr.omean) y = (y - tr.omean[c]) / tr.ostd[c];
      d = O[rr * n.op + c] - y;
      g = 2.f * tr.scale * d;
    }
    O[rr * n.op + c] = d;
    uint16_t gb = f2bf(g);
    D3[rr * l3 + c] = gb;
    tr.d3t[(size_t)c * tr.rp + r] = gb;
    tr.f3[(size_t)c * tr.rp + r] = g;
  }
  __syncthreads();
  if (tid < FROWS) {
    float l = 0.f;
    if (r0 + tid < tr.rvalid)
      for (int c = 0; c < n.nout; c++) { float d = O[tid * n.op + c]; l += d * d; }
    tr.rowloss[r0 + tid] = l;
  }
  net_mm<NT, PF>(acc, b, D3, l3, n.W3, n.op, ht, wave, lane);
  net_load<NT, PF>(b, n.W2, n.nh, ht, wave, lane, 0);
  net_back<NT>(acc, z2, ht, wave, lane, H2, lh, tr.d2t, tr.f2, tr.rp, r0);
  __syncthreads();
  net_mm<NT, PF>(acc, b, H2, lh, n.W2, n.nh, ht, wave, lane);
  net_back<NT>(acc, z1, ht, wave, lane, nullptr, 0, tr.d1t, tr.f1, tr.rp, r0);
}

// One weight matrix's gradient a^T b: a [M][K], b [N][K] (bf16, K = batch
// rows), K cut into slices of kchunk rows whose sums are added in order; its
// workgroups are blk0 .. of the launch, one per 16 x 32 tile
struct WgMat { const uint16_t *a, *b; int M, N, kchunk, blk0; size_t off; };
// One bias gradient: the row sums of f [C][K] in slices of 128; workgroups from blk0, eight columns each
struct WgBias { const float* f; int C, blk0; size_t off; };
struct WgArgs {
  WgMat w[3];
  WgBias b[3];
  int K;
  // update: AdamW on p (m, v) and the bf16 copies pb, pbt; else the gradient into g
  int update;
  float *p, *g, *m, *v;
  uint16_t *pb, *pbt;
  float lr, b1, b2, eps, wd, c1, c2;
};

__device__ __forceinline__ float wg_update(const WgArgs& A, size_t i, float gi) {
  float mi = A.m[i], vi = A.v[i];
  float pi = adamw_step(A.p[i], gi, mi, vi, A.lr, A.b1, A.b2, A.eps, A.wd, A.c1, A.c2);
  A.m[i] = mi;
  A.v[i] = vi;
  A.p[i] = pi;
  return pi;
}

// One 16 x 32 tile of a weight gradient per workgroup (256 for 195-256-256-18,
// one per CU, and 68 of bias columns after them): each wave forms the sums of its slices of K, 4 K steps of loads
// ahead of the products, and leaves them in LDS, where a thread per entry adds
// the slices in order and applies the update; no partial tile goes through
// memory. Column tiles are the fastest index, so that an XCD (workgroup index
// mod 8) reads an eighth of b, not all of it, beside a. A batch of
// 4096 x 195-256-256-18, 16 x 16 tiles with their whole K in one wave (512
// waves, a chain of 128 steps) -> this: 34.6 -> 23.0 us.
enum { WSL = 32, WTHREADS = 512, WWAVES = WTHREADS / 64 };
__global__ void __launch_bounds__(WTHREADS) k_wgrad(WgArgs A) {
  __shared__ __align__(16) float part[WSL][512];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, blk = blockIdx.x, K = A.K;
  if (blk < A.b[0].blk0) {
    int q = blk >= A.w[2].blk0 ? 2 : (blk >= A.w[1].blk0 ? 1 : 0);
    const WgMat& w = A.w[q];
    int nt = w.N / 32, k = blk - w.blk0, mi = k / nt, ni = k - mi * nt;
    const uint16_t* pa = w.a + (size_t)(16 * mi + (lane & 15)) * K + 8 * (lane >> 4);
    const uint16_t* pb = w.b + (size_t)(32 * ni + (lane & 15)) * K + 8 * (lane >> 4);
    const size_t col16 = (size_t)16 * K;
    constexpr int PF = 4;
    const int KS = K / 32, sl = w.kchunk / 32, nsl = (KS + sl - 1) / sl;
    float s = 0.f;
    for (int p0 = 0; p0 < nsl; p0 += WSL) {
      // this wave's slices p0 + wave, + 8, ..: their K steps as one sequence of
      // groups of PF (a slice's last group may be short)
      int pe = p0 + WSL < nsl ? p0 + WSL : nsl, gps = (sl + PF - 1) / PF;
      int ng = p0 + wave < pe ? ((pe - 1 - p0 - wave) / WWAVES + 1) * gps : 0;
      v8bf a0[PF], b0[2 * PF], a1[PF], b1[2 * PF];
      v4f acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
      auto range = [&](int g, int& slice, int& k0, int& n) {
        int j = g / gps, o = (g - j * gps) * PF;
        slice = p0 + wave + WWAVES * j;
        k0 = slice * sl + o;
        int e = (slice + 1) * sl < KS ? (slice + 1) * sl : KS;
        n = e - k0;  // <= 0: nothing left of a short last slice
      };
      auto load = [&](v8bf (&av)[PF], v8bf (&bv)[2 * PF], int g) {
        if (g >= ng) return;
        int slice, k0, n;
        range(g, slice, k0, n);
#pragma unroll
        for (int i = 0; i < PF; i++)
          if (i < n) {
            av[i] = *reinterpret_cast<const v8bf*>(pa + 32 * (k0 + i));
            bv[i] = *reinterpret_cast<const v8bf*>(pb + 32 * (k0 + i));
            bv[PF + i] = *reinterpret_cast<const v8bf*>(pb + col16 + 32 * (k0 + i));
          }
      };
      auto mma = [&](const v8bf (&av)[PF], const v8bf (&bv)[2 * PF], int g) {
        if (g >= ng) return;
        int slice, k0, n;
        range(g, slice, k0, n);
#pragma unroll
        for (int i = 0; i < PF; i++)
          if (i < n) {
            acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bv[i], acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bv[PF + i], acc1, 0, 0, 0);
          }
        if (g % gps == gps - 1) {
          *reinterpret_cast<v4f*>(&part[slice - p0][4 * lane]) = acc0;
          *reinterpret_cast<v4f*>(&part[slice - p0][256 + 4 * lane]) = acc1;
          acc0 = acc1 = v4f{0.f, 0.f, 0.f, 0.f};
        }
      };
      load(a0, b0, 0);
      for (int g = 0; g < ng; g += 2) {
        load(a1, b1, g + 1);
        mma(a0, b0, g);
        load(a0, b0, g + 2);
        mma(a1, b1, g + 1);
      }
      __syncthreads();
      for (int i = 0; i < pe - p0; i++) s += part[i][tid];
      __syncthreads();
    }
    // thread tid: entry i = tid % 4 of lane l of the tile's left or right half
    int l = (tid >> 2) & 63, m = 16 * mi + 4 * (l >> 4) + (tid & 3), n = 32 * ni + 16 * (tid >> 8) + (l & 15);
    size_t e = w.off + (size_t)m * w.N + n;
    if (A.update) {
      uint16_t pv = f2bf(wg_update(A, e, s));
      A.pb[e] = pv;
      A.pbt[w.off + (size_t)n * w.M + m] = pv;
    } else {
      A.g[e] = s;
    }
    return;
  }
  // a bias: eight columns, 64 slices of 128 rows at a time; a slice is summed in
  // four interleaved chains, the slices in four more
  int q = blk >= A.b[2].blk0 ? 2 : (blk >= A.b[1].blk0 ? 1 : 0);
  const WgBias& bi = A.b[q];
  int c = WWAVES * (blk - bi.blk0) + wave, nsl = (K + 127) / 128;
  float run = 0.f;
  for (int s0 = 0; s0 < nsl; s0 += 64) {
    float c0 = 0.f, c1 = 0.f, c2 = 0.f, c3 = 0.f;
    if (c < bi.C && s0 + lane < nsl) {
      int ra = 128 * (s0 + lane), rb = ra + 128 < K ? ra + 128 : K;
      const float* f = bi.f + (size_t)c * K;
      int r = ra;
      for (; r + 64 <= rb; r += 64) {  // 16 loads in flight: the kernel 23.0 -> 21.7 us
        float4 v[16];
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = *reinterpret_cast<const float4*>(f + r + 4 * i);
#pragma unroll
        for (int i = 0; i < 16; i++) { c0 += v[i].x; c1 += v[i].y; c2 += v[i].z; c3 += v[i].w; }
      }
      for (; r < rb; r += 4) {
        float4 v = *reinterpret_cast<const float4*>(f + r);
        c0 += v.x; c1 += v.y; c2 += v.z; c3 += v.w;
      }
    }
    part[wave][lane] = (c0 + c1) + (c2 + c3);
    __syncthreads();
    int e = nsl - s0 < 64 ? nsl - s0 : 64;
    if (lane < 4)
      for (int k = lane; k < e; k += 4) run += part[wave][k];
    __syncthreads();
  }
  if (lane < 4) part[wave][lane] = run;
  __syncthreads();
  if (lane == 0 && c < bi.C) {
    float g = (part[wave][0] + part[wave][1]) + (part[wave][2] + part[wave][3]);
    if (A.update) wg_update(A, bi.off + c, g);
    else A.g[bi.off + c] = g;
  }
}

// bf16 copies of the weights in both orders (weights outside k_wgrad's updates)
struct ShadowArgs { size_t off[3]; int rows[3], cols[3]; };
__global__ void k_shadow(ShadowArgs a, const float* __restrict__ p, uint16_t* __restrict__ pb, uint16_t* __restrict__ pbt) {
  int q = blockIdx.y, i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.rows[q] * a.cols[q]) return;
  uint16_t v = f2bf(p[a.off[q] + i]);
  pb[a.off[q] + i] = v;
  int r = i / a.cols[q], c = i - r * a.cols[q];
  pbt[a.off[q] + (size_t)c * a.rows[q] + r] = v;
}
