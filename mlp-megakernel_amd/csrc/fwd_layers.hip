// Forward for the networks the megakernels do not take (16-bit tensors, widths
// up to 512, up to 8 layers): every layer of a row tile in one launch, the
// activations in LDS, the weights read from L2 in MFMA operand order.
//
// The reference's kernel takes any hidden width as constexpr tile loops
// (/root/reference/kernel.py:60-123, README.md:62,68).  From H = 272 on, a
// row block's activations no longer fit a wave's registers beside its
// accumulators (fwd_wide.h), and such networks ran as fp32 library GEMMs with
// the conversions and the softplus as launches of their own: 128-512-512-128
// at 16,384 rows 182 us, of which 121 us fp32 GEMMs (the fp32 matrix rate is
// a ninth of the 16-bit one, and a 16-bit product is exact in fp32 either
// way).
//
//  * pack_kernel writes the weights once per call into the caller's workspace
//    as MFMA A operands (1 KiB fragments: 32 features x 16 inputs, 16 bytes
//    per lane), both dimensions padded with zeros to multiples of 64: the
//    main kernel then reads a fragment with one 16-byte load per lane, and
//    needs no test of a width in its loop.  (Read straight from the row-major
//    W_l, a lane's eight inputs of one feature are eight loads; at 256-wide
//    layers these were 20 % of such a kernel's time.)  Both launches at that
//    size: 25.4 us per call, 4.4 us of it the packing.
//  * fwd_layers_kernel: a workgroup of 8 waves owns a tile of 32 RB rows, in
//    one LDS tile of 16-bit activations that the layers overwrite in turn.
//    Wave f computes output features [64 f, 64 f + 64) of every row; a layer
//    of at most 256 features splits the rows over the waves as well, so every
//    fragment is read by one wave, or by the few that share its rows.  (Of a
//    layer of at most 64 features two waves have work, the others wait: 0.12 ns
//    per row and layer whatever its width.)
//  * Softplus as max(z, 0) + log1p(e^-|z|) in fp32, handed on rounded to the
//    tensor format as the reference rounds its h (kernel.py:110); the stash is
//    that fp32 value.
#include "device_common.h"
#include "host_common.h"
#include "params.h"

namespace mlpmk {
namespace layers {

constexpr int kMaxWidth = 512;
constexpr int NWV = 8;                  // waves per workgroup
constexpr int kChunks = kMaxWidth / 8;  // 16-byte pieces of a tile row
constexpr int kDepth = 4;               // K-steps of weights in flight

struct Params {
  const f16* x;
  f16* out;
  const f16* w[kMaxLayersHost];     // packed: layer l's fragments, (pad64(out) / 32) blocks of pad64(in) / 16 K-steps
  float* stash[kMaxLayersHost];     // stash[l] = h_{l+1}, fp32 [M, d[l+1]], or null
  int64_t M;
  int L;
  int dims[kMaxLayersHost + 1];
};

__host__ __device__ constexpr int pad64(int n) { return (n + 63) & ~63; }

// softplus(z) = max(z, 0) + log1p(y), y = e^-|z|: two transcendentals and
// ten more operations.
//  * y = 2^p e^r with p = -|z| log2 e rounded and r = -|z| - p ln 2 (ln 2 in two
//    parts), e^r = 1 + r: without r the rounding of p alone moves y by
//    |z| 2^-24 (3.8e-6 at z = -80; the stash is fp32, and the elementwise
//    kernel of the layer-by-layer route carries the same correction).
//  * log1p(y) = ln 2 log2(w) + (y - (w - 1)) with w = 1 + y rounded: the second
//    term is what the rounding of w dropped (its factor 1 / w is left out: the
//    term is below 2^-24 where w is not close to 1), so small y keep their
//    digits.
// y is clamped to [0, 1], which makes the NaN (inf - inf) of an infinite z 0 and
// takes no operation of its own (the multiply-add's output modifier); a NaN z
// comes through the maximum.  Largest relative error, here
// / elementwise kernel / without r: 1.4e-7 / 1.9e-7 / 3.9e-6 for z in [-87, -20],
// 2.9e-7 / 3.5e-7 / 1.1e-6 in [-20, -5], 2.7e-7 / 3.3e-7 / 4.4e-7 above.  r takes
// three operations: 128-512-512-128 at 16,384 rows 24.0 -> 25.4 us.
constexpr float kLn2Lo = -1.904654323148236e-9f;  // ln 2 - kLn2
__device__ __forceinline__ float softplus_n(float z) {
  const float a = -__builtin_fabsf(z), p = a * kLog2e, e = __builtin_amdgcn_exp2f(p);
  const float r = __builtin_fmaf(p, -kLn2Lo, __builtin_fmaf(p, -kLn2, a));
  const float y = __builtin_amdgcn_fmed3f(__builtin_fmaf(e, r, e), 0.0f, 1.0f);
  const float w = 1.0f + y;
  const float c = y - (w - 1.0f);
  return __builtin_elementwise_maximum(z, 0.0f) + __builtin_fmaf(kLn2, __builtin_amdgcn_logf(w), c);
}

// Packs every layer: thread (l, fragment, lane) writes its 16 bytes.  Lane
// (i, g) of fragment (mb, s): W_l[16 s + 8 g + j][outfeat(mb, i)], j = 0..7.
struct PackParams {
  const f16* w[kMaxLayersHost];
  int64_t first[kMaxLayersHost + 1];  // first fragment lane of layer l
  f16* dst;
  int L;
  int dims[kMaxLayersHost + 1];
};
__global__ __launch_bounds__(256) void pack_kernel(PackParams p) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= p.first[p.L]) return;
  int l = 0;
  while (l + 1 < p.L && t >= p.first[l + 1]) ++l;
  const int K = p.dims[l], N = p.dims[l + 1], KS = pad64(K) / 16;
  const int item = (int)(t - p.first[l]), fr = item >> 6, lane = item & 63;
  const int col = outfeat(fr / KS, lane & 31), k0 = 16 * (fr % KS) + 8 * (lane >> 5);
  f16x8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = (col < N && k0 + j < K) ? p.w[l][(int64_t)(k0 + j) * N + col] : (f16)0.0f;
  *reinterpret_cast<f16x8*>(p.dst + t * 8) = v;
}

// LDS slot (16-byte units) of (row, piece): the XOR spreads the same piece of
// eight consecutive rows over distinct banks.
__device__ __forceinline__ int tslot(int row, int piece) { return row * kChunks + (piece ^ (row & 7)); }

constexpr uint32_t kOut = 0x80000000u;  // an offset past every resource: loads read zeros, stores are dropped

template <int RB, bool BF, bool STASH>
struct Wave {
  static constexpr int ROWS = 32 * RB;
  const Params& p;
  i32x4* tile;  // [ROWS][kChunks]
  int lane, n, g, wv;
  int64_t row0;
  i32x4 wb[kDepth][2];  // fragments of the next K-steps: features [64 f, + 32) and [64 f + 32, + 32)

  // A wave's share of a layer of N features: feature group f and row part
  // `part` of `split` (split > 1 when the layer has at most half the waves'
  // features).
  struct Share {
    int f, part, split;
  };
  __device__ __forceinline__ Share share(int N) const {
    int split = 1;
    while (split < NWV && 64 * (NWV / (2 * split)) >= N) split *= 2;
    const int groups = NWV / split;
    return Share{wv % groups, wv / groups, split};
  }
  __device__ __forceinline__ uint32_t rows_left() const {
    const int64_t left = p.M - row0;
    return (uint32_t)(left < ROWS ? (left > 0 ? left : 0) : ROWS);
  }
  // Feature group f of layer l: its two blocks' fragments, K-step s at
  // byte 1024 s (+ 1024 KS for the second block).  A group past the layer's
  // features has an empty resource.
  __device__ __forceinline__ rsrc_t wrsrc(int l, int f) const {
    const int KS = pad64(p.dims[l]) / 16;
    const bool any = 64 * f < p.dims[l + 1];
    return make_rsrc(p.w[l] + (int64_t)f * 2 * KS * 512, any ? (uint32_t)KS * 2048u : 0u);
  }
  __device__ __forceinline__ void load_w(const rsrc_t& r, int KS, int s, int t) {
    const int o = s * 1024 + lane * 16;
    wb[t][0] = __builtin_amdgcn_raw_buffer_load_b128(r, s < KS ? o : (int)kOut, 0, 0);
    wb[t][1] = __builtin_amdgcn_raw_buffer_load_b128(r, s < KS ? o + KS * 1024 : (int)kOut, 0, 0);
  }
  __device__ __forceinline__ void request(int l) {
    const rsrc_t r = wrsrc(l, share(p.dims[l + 1]).f);
    const int KS = pad64(p.dims[l]) / 16;
#pragma unroll
    for (int t = 0; t < kDepth; ++t) {
      load_w(r, KS, t, t);
      __builtin_amdgcn_sched_barrier(0);  // in this order: the K loop counts them
    }
  }

  // x rows of the tile, features padded with zeros to whole K turns, 128
  // features of every row in flight.
  __device__ __forceinline__ void load_x() {
    const int D = p.dims[0];
    const rsrc_t r = make_rsrc(p.x + row0 * D, rows_left() * (uint32_t)D * 2u);
    constexpr int U = (ROWS * 8 + NWV * 64 - 1) / (NWV * 64);
    const int tid = wv * 64 + lane, row = tid >> 3;
    for (int c = tid & 7; 8 * c < pad64(D); c += 16) {
      i32x4 v[2][U];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int rr = row + u * 8 * NWV, cc = c + 8 * h;
          v[h][u] = __builtin_amdgcn_raw_buffer_load_b128(
              r, rr < ROWS && 8 * cc < D ? (rr * D + 8 * cc) * 2 : (int)kOut, 0, 0);
        }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int rr = row + u * 8 * NWV, cc = c + 8 * h;
          if (rr < ROWS && 8 * cc < pad64(D)) tile[tslot(rr, cc)] = v[h][u];
        }
    }
  }

  // Layer l for this wave's RBW row blocks from block rb0 and feature group
  // f; `next` is the layer whose first weights to request (-1: none).
  template <int RBW>
  __device__ __forceinline__ void layer(int l, int f, int rb0, bool active, int next) {
    const int N = p.dims[l + 1];
    f32x16 acc[2][RBW] = {};
    if (active) {
      const rsrc_t r = wrsrc(l, f);
      const int KS = pad64(p.dims[l]) / 16;
      int sl[RBW];
#pragma unroll
      for (int b = 0; b < RBW; ++b) sl[b] = (32 * (rb0 + b) + n) * kChunks;
      const int x7 = n & 7;
      f16x8 in[2][RBW];
#pragma unroll
      for (int b = 0; b < RBW; ++b) in[0][b] = __builtin_bit_cast(f16x8, tile[sl[b] + (g ^ x7)]);
      // K-step t of a turn: the reads of the next K-step's activations go out
      // first, then its MFMAs with the weight requests kDepth K-steps ahead
      // among them.  The fences keep the reads a K-step ahead; left alone, the
      // scheduler puts each right before its MFMA.
      for (int c = 0; c < KS; c += kDepth) {
#pragma unroll
        for (int t = 0; t < kDepth; ++t) {
          const int s1 = c + t + 1 < KS ? c + t + 1 : 0;  // (past the last one: piece 0 again)
#pragma unroll
          for (int b = 0; b < RBW; ++b)
            in[(t + 1) & 1][b] = __builtin_bit_cast(f16x8, tile[sl[b] + ((2 * s1 + g) ^ x7)]);
          const f16x8 a0 = __builtin_bit_cast(f16x8, wb[t][0]), a1 = __builtin_bit_cast(f16x8, wb[t][1]);
#pragma unroll
          for (int b = 0; b < RBW; ++b) {
            acc[0][b] = mfma32x32x16<BF>(a0, in[t & 1][b], acc[0][b]);
            acc[1][b] = mfma32x32x16<BF>(a1, in[t & 1][b], acc[1][b]);
          }
          load_w(r, KS, c + kDepth + t, t);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (next >= 0) request(next);
    // Registers 0..7 of block q: features 64 f + 32 q + 8 g + [0..7]; 8..15: + 16.
    if (l + 1 < p.L) {
      f16x8 h16[RBW][4];
      if (active) {
        rsrc_t sr;
        if constexpr (STASH)  // (an entry not requested: an empty resource, its stores dropped)
          sr = make_rsrc(p.stash[l] + row0 * N, p.stash[l] ? rows_left() * (uint32_t)N * 4u : 0u);
#pragma unroll
        for (int b = 0; b < RBW; ++b)
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            float h[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) h[j] = softplus_n(acc[a >> 1][b][8 * (a & 1) + j]);
            h16[b][a] = pack8<BF>(h[0], h[1], h[2], h[3], h[4], h[5], h[6], h[7]);
            if constexpr (STASH) {
              const int cc = 64 * f + 16 * a + 8 * g;
              const uint32_t e = cc < N ? (uint32_t)((32 * (rb0 + b) + n) * N + cc) * 4u : kOut;  // dropped past N
              buf_store16<kStashStore>((f32x4){h[0], h[1], h[2], h[3]}, sr, e);
              buf_store16<kStashStore>((f32x4){h[4], h[5], h[6], h[7]}, sr, e + 16);
            }
          }
      }
      // Features that only pad the layer (softplus(0), or NaN where a row holds
      // an infinity: inf * 0) are handed on as zeros, against zero weights.  A
      // piece of 8 is a feature of the layer or past it as a whole.
      if (active && 64 * f + 64 > N) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const bool past = 64 * f + 16 * a + 8 * g >= N;
#pragma unroll
          for (int b = 0; b < RBW; ++b) h16[b][a] = past ? f16x8{} : h16[b][a];
        }
      }
      __syncthreads();  // every wave has read the layer's inputs
      if (active) {
#pragma unroll
        for (int b = 0; b < RBW; ++b)
#pragma unroll
          for (int a = 0; a < 4; ++a)
            tile[tslot(32 * (rb0 + b) + n, 8 * f + 2 * a + g)] = __builtin_bit_cast(i32x4, h16[b][a]);
      }
    } else if (active) {
      const rsrc_t orr = make_rsrc(p.out + row0 * N, rows_left() * (uint32_t)N * 2u);
#pragma unroll
      for (int b = 0; b < RBW; ++b)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const int cc = 64 * f + 16 * a + 8 * g;
          const uint32_t e = (uint32_t)((32 * (rb0 + b) + n) * N + cc);
          float v[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = acc[a >> 1][b][8 * (a & 1) + j];
          if (N % 8 == 0) {
            // Rows of up to 1 KiB written a piece at a time: L2 merges them.
            buf_store16<kStashStore>(pack8<BF>(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]), orr,
                                     cc < N ? e * 2 : kOut);
          } else {
            // Each element converted on its own (taken out of a packed
            // vector, the 2-byte store builtin was given element 0 every time).
#pragma unroll
            for (int j = 0; j < 8; ++j)
              __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, f32_to_elem<BF>(v[j])), orr,
                                                    (int)(cc + j < N ? (e + j) * 2 : kOut), 0, kStashStore);
          }
        }
    }
    __syncthreads();  // hidden layer: the tile holds its output; last layer: the tile is free
  }

  template <int RBW = RB>
  __device__ __forceinline__ void layer_split(int l, const Share& sh, int next) {
    // (Less than one row block per wave: the first RB parts take one each.)
    if constexpr (RBW > 1) {
      if (sh.split * RBW > RB) {
        layer_split<RBW / 2>(l, sh, next);
        return;
      }
    }
    layer<RBW>(l, sh.f, sh.part * RBW, sh.part * RBW < RB && 64 * sh.f < p.dims[l + 1], next);
  }
};

template <int RB, bool BF, bool STASH>
__global__ __launch_bounds__(NWV * 64) void fwd_layers_kernel(Params p) {
  using W = Wave<RB, BF, STASH>;
  __shared__ i32x4 tile[W::ROWS * kChunks];
  const int lane = threadIdx.x & 63;
  W w{p, tile, lane, lane & 31, lane >> 5, __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), 0};
  const int64_t ntiles = (p.M + W::ROWS - 1) / W::ROWS;
  int64_t t = blockIdx.x;
  if (t >= ntiles) return;  // the whole workgroup
  w.request(0);
  for (; t < ntiles; t += gridDim.x) {
    w.row0 = t * W::ROWS;
    w.load_x();
    __syncthreads();
    for (int l = 0; l < p.L; ++l)
      w.template layer_split<>(l, w.share(p.dims[l + 1]), l + 1 < p.L ? l + 1 : (t + gridDim.x < ntiles ? 0 : -1));
  }
}

template <int RB, bool BF, bool STASH>
static int launch(const Params& p, int cus, hipStream_t st) {
  const void* kern = reinterpret_cast<const void*>(&fwd_layers_kernel<RB, BF, STASH>);
  constexpr int kMaxDev = 64;
  static int occ_cache[kMaxDev];  // 0 = unknown; benign race (idempotent value)
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  int occ = (dev >= 0 && dev < kMaxDev) ? occ_cache[dev] : 0;
  if (occ <= 0) {
    const int rc = kernel_occupancy(kern, NWV * 64, &occ);
    if (rc != MLPMK_OK) return rc;
    if (dev >= 0 && dev < kMaxDev) occ_cache[dev] = occ;
  }
  const int64_t ntiles = (p.M + 32 * RB - 1) / (32 * RB), cap = (int64_t)cus * occ;
  hipLaunchKernelGGL((fwd_layers_kernel<RB, BF, STASH>), dim3((unsigned)(ntiles < cap ? ntiles : cap)), dim3(NWV * 64),
                     0, st, p);
  e = hipGetLastError();
  return e == hipSuccess ? MLPMK_OK : hip_fail(e, "fwd layers kernel launch");
}

template <int RB>
static int launch_any(const Params& p, bool bf, bool stash, int cus, hipStream_t st) {
  if (bf) return stash ? launch<RB, true, true>(p, cus, st) : launch<RB, true, false>(p, cus, st);
  return stash ? launch<RB, false, true>(p, cus, st) : launch<RB, false, false>(p, cus, st);
}

}  // namespace layers

// 16-bit networks of 2..8 layers, input and hidden widths multiples of 8 in
// [8, 512], output width in [1, 512].
bool fwd_layers_supported(int L, const int* dims, int dtype) {
  if (L < 2 || L > kMaxLayersHost || (dtype != MLPMK_DTYPE_F16 && dtype != MLPMK_DTYPE_BF16)) return false;
  for (int i = 0; i < L; ++i)
    if (dims[i] < 8 || dims[i] > layers::kMaxWidth || dims[i] % 8 != 0) return false;
  return dims[L] >= 1 && dims[L] <= layers::kMaxWidth;
}

// The packed weights.
int64_t fwd_layers_workspace(int L, const int* dims) {
  int64_t b = 0;
  for (int l = 0; l < L; ++l) b += (int64_t)layers::pad64(dims[l]) * layers::pad64(dims[l + 1]) * 2;
  return b;
}

int fwd_layers_dispatch(int L, const int* dims, const FwdParams& fp, bool stash, int dtype, void* ws, hipStream_t st) {
  int cus = 0;
  const int rc = current_device_cus(&cus);
  if (rc != MLPMK_OK) return rc;
  layers::PackParams pk = {};
  layers::Params p = {};
  p.x = fp.x;
  p.out = fp.out;
  p.M = fp.M;
  p.L = pk.L = L;
  pk.dst = static_cast<f16*>(ws);
  int64_t o = 0;
  for (int l = 0; l < L; ++l) {
    pk.w[l] = fp.w[l];
    pk.first[l] = o;
    p.w[l] = pk.dst + o * 8;
    p.stash[l] = fp.stash[l];
    o += (int64_t)layers::pad64(dims[l]) * layers::pad64(dims[l + 1]) / 8;
  }
  pk.first[L] = o;
  for (int l = 0; l <= L; ++l) p.dims[l] = pk.dims[l] = dims[l];
  (void)hipGetLastError();
  hipLaunchKernelGGL(layers::pack_kernel, dim3((unsigned)((o + 255) / 256)), dim3(256), 0, st, pk);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "weight packing kernel launch");
  const bool bf = dtype == MLPMK_DTYPE_BF16;
  // Tiles of 64 rows as soon as tiles of 32 would give a CU a second one.  Up to
  // 64 rows per CU that leaves CUs without a tile, but each reads the weights
  // once where two tiles read them twice (64-row / 32-row tiles, us, replayed
  // graph, 256 CUs): 128-512-512-128 at 9,000 rows 24.1 / 27.3, 16,000 25.6 / 28.8;
  // 512-512-512-512-512 41.8 / 51.3, 49.8 / 59.3; 6 x 128 20.5 / 23.7, 20.9 / 24.0;
  // 8 x 32 21.5 / 21.6; only 128-320-320-128 is better off in two: 20.9 / 19.5,
  // 21.4 / 19.0 (five feature groups of eight waves).
  return fp.M > (int64_t)32 * cus ? layers::launch_any<2>(p, bf, stash, cus, st)
                                  : layers::launch_any<1>(p, bf, stash, cus, st);
}

}  // namespace mlpmk
