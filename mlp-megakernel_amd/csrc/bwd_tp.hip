// Two-pass backward for gfx950 (MI355X): the training backward of the
// softplus MLP as a data-gradient pass spread over the whole chip, then a
// weight-gradient pass whose workgroups each own a block of dW.
//
// Replaces the same reference interface as bwd.hip -- the fused backward of
// the FusedMLPSoftplus autograd function (/root/reference/mlp_fused.md:80-112,
// README.md:30-32) -- for the cases the one-pass megakernel does not serve
// well or at all:
//
//  * small batches (a few thousand rows): the one-pass kernel keeps a whole
//    dW per workgroup, so it runs one 128-row round per workgroup on M / 128
//    CUs (32 of 256 at M = 4096) and then reduces 192 KiB of partials per
//    workgroup;
//  * fp32 tensors (the reference's INPUT_DTYPE = fp32 kernels,
//    mlp_fused.md:159-166): every operand is split into bf16 hi + lo
//    (hi = bf16(v), lo = bf16(v - hi)) and each product is hi*hi + hi*lo +
//    lo*hi on the bf16 MFMA -- fp32's exponent range and a ~16-bit
//    significand (the lo*lo term, below 2^-16 relative, is dropped), where
//    the reference's TF32 operands keep 10 bits;
//  * widths above 128 (up to 256; the reference lists larger H as its next
//    step, mlp_fused.md:453-454), whose dgrad weights and exchange tiles do
//    not fit one workgroup's LDS beside a whole dW of accumulators.
//
// Math (mlp_fused.md:88-95), a_0 = x, a_l = h_l from the fp32 stash,
// dz_{L-1} = dL/dout:
//     dz_{l-1} = (dz_l . W_l^T) * (1 - exp(-h_l)),   dx = dz_0 . W_0^T
//     dW_l     = a_l^T . dz_l
//
// Pass 1, tp_dgrad_kernel (persistent over tiles of 32 or 64 rows): wave w owns
// output features [32w, 32w + 32) of every data-gradient layer, with its A
// fragments (16 contiguous bytes of a W_l row per lane) loaded once into
// registers for the 3-layer 128-wide network and read from L2 otherwise;
// layers hand dz between waves through two LDS tiles, and every dz_{l-1},
// l >= 1, is also written to the workspace.  The next tile's rows are
// requested while this one computes.  When dw is to be written
// (MLPMK_BWD_WRITE_DW) this pass also clears it.  At M = 4096 that is 128
// workgroups each running a chain of 8-MFMA steps, instead of 32 running
// whole 128-row rounds.
//
// Pass 2, tp_wgrad_kernel: a workgroup owns a TQI x TQO block of 64 x 64
// "quads" of one dW_l and a chunk of rows; it stages a_l (from x or the
// stash) and dz_l (from dL/dout or the workspace) as 16-bit tiles
// [row][feature] in LDS, and its waves read both MFMA operands with the
// transposing ds_read_b64_tr_b16, as bwd.hip's wgrad does.  Its sums go to dw
// as fp32 atomics at the end (measured at M = 4096 / 16384: 14.2 / 24.1 us per
// backward, against 16.4 / 31.0 us with per-chunk partial sums and a combine
// kernel).  The summation order of dw is therefore not fixed.
//
// Where it runs (bwd.hip, bwd_path): fp32 tensors and widths above 128
// always; the 16-bit networks the one-pass megakernel also serves up to
// MLPMK_TP_MAX_ROWS rows (3L-128, MI355X, per backward call as a replayed
// graph, two-pass vs one-pass: 14.2 vs 23.0 us at 4096 rows, 24.1 vs 26.8 at
// 16384, with dx 49.0 vs 34.3 at 32768).
#include <type_traits>

#include "device_common.h"
#include "host_common.h"
#include "params.h"
#include "tp_common.h"

namespace mlpmk {

namespace tp {

// ---------------------------------------------------------------------------
// Pass 1: data gradients
// ---------------------------------------------------------------------------

template <class N, bool DX>
struct DgGeo {
  static constexpr int L = N::L;
  static constexpr int LO = DX ? 0 : 1;  // lowest layer with a data gradient
  static constexpr int blocks(int l) { return (N::d[l] + 31) / 32; }
  static constexpr int ks(int l) { return N::d[l + 1] / 16; }  // K-steps: features of dz_l
  static constexpr int nwv() {
    int m = 1;
    for (int l = LO; l < L; ++l) m = blocks(l) > m ? blocks(l) : m;
    return m;
  }
  static constexpr int ksm() {
    int m = 1;
    for (int l = LO; l < L; ++l) m = ks(l) > m ? ks(l) : m;
    return m;
  }
  // Exchange tile width (features per row; a power of two for the swizzle, of
  // whole 64-feature K turns): dL/dout (d[L] features), and layer l >= LO + 1
  // hands dz_{l-1} (d[l] features) to layer l - 1.
  static constexpr int tw() {
    int m = 64;
    while (m < N::d[L]) m *= 2;
    for (int l = LO + 1; l < L; ++l)
      while (m < N::d[l]) m *= 2;
    return m;
  }
  static constexpr int NWV = nwv(), KSM = ksm(), TW = tw(), CH = TW / 8;
  static constexpr bool valid() {
    for (int i = 0; i <= L; ++i)
      if (N::d[i] > 256 || N::d[i] % 16 != 0) return false;
    return L >= 2 && NWV <= 8;
  }
};

// Packed weights of a layer (16-bit tensors): fragment (mb, s), 1 KiB, holds in
// lane (i, g) W_l[outfeat(mb, i)][16s + 8g + 0..7]; K-steps padded with zeros
// to whole turns of 4.
__host__ __device__ constexpr int pack_ks(int nout) { return (nout + 63) / 64 * 4; }
__host__ __device__ constexpr int pack_frags(int k, int nout) { return (k + 31) / 32 * pack_ks(nout); }
struct PackParams {
  const f16* w[kMaxLayersHost];
  f16* dst[kMaxLayersHost];
  int first[kMaxLayersHost + 1];  // first fragment lane of layer l
  int dims[kMaxLayersHost + 1];
  int L;
};
__global__ __launch_bounds__(256) void tp_pack_kernel(PackParams p) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= p.first[p.L]) return;
  int l = 0;
  while (l + 1 < p.L && t >= p.first[l + 1]) ++l;
  const int K = p.dims[l], Nout = p.dims[l + 1], KP = pack_ks(Nout);
  const int item = t - p.first[l], f = item >> 6, lane = item & 63;
  const int row = outfeat(f / KP, lane & 31), c = 16 * (f % KP) + 8 * (lane >> 5);
  // (widths here are multiples of 8: a piece lies in the row or past it)
  f16x8 v = {};
  if (row < K && c < Nout) v = *reinterpret_cast<const f16x8*>(p.w[l] + (int64_t)row * Nout + c);
  *reinterpret_cast<f16x8*>(p.dst[l] + (int64_t)item * 8) = v;
}

// A workgroup of NWV waves runs tiles of 32 RB rows, one after the other; wave w
// owns features [32w, 32w + 32) of every data gradient and all rows of the
// tile.  dL/dout and every dz_l go through LDS tiles (two, in turns: one
// barrier per layer), from which each wave reads its B operands a K-step ahead
// of the MFMA that takes them.  Everything that comes from memory is requested
// a tile ahead: the next tile's dL/dout (each thread a share of it) right after
// this tile's went into LDS, the next tile's h_l into the registers that this
// tile's sigma(h_l) just left.
//
// RES: every layer's fragments stay in registers for the whole kernel
// (loaded once per workgroup); otherwise they are read from L2 through a ring
// of kRing K-steps, the next layer's first ones requested before this layer's
// results are evaluated.  PK: from the packed copy (tp_pack_kernel), 1 KiB
// whole; from W_l itself a fragment is 32 bytes of each of 32 rows, and at
// width 256 the 8 waves' rows do not stay in the vector cache until the
// K-steps that use the rest of their lines (128-256-256-128 bf16 at 100,003
// rows: this pass 101 -> 80 us, the packing 4.7).
template <class N, int EM, bool DX, bool RES, int RB, bool PK>
struct DgWave {
  using G = DgGeo<N, DX>;
  static constexpr int L = N::L, CH = G::CH, NT = EM == EM_F32 ? 2 : 1;
  static constexpr int ROWS = 32 * RB;
  static constexpr int kRing = 4;
  static constexpr uint32_t kPast = 0x80000000u;  // past every resource: loads read zeros
  // dL/dout pieces (8 elements) of a tile per thread.
  static constexpr int OCH = (N::d[L] + 63) / 64 * 8;  // pieces of a row, padded to whole K turns
  static constexpr int PD = (ROWS * OCH + G::NWV * 64 - 1) / (G::NWV * 64);
  struct Raw {  // 8 tensor elements as loaded
    f32x4 v[NT];
  };
  const TpParams& p;
  f16x8 (*tile)[NT][ROWS * CH];  // [2][NT][ROWS * CH]
  int lane, n, g, w;
  int par = 0;                          // tile of the next hand-over
  Opnd fr[RES ? L : 1][RES ? G::KSM : 1];  // RES: this wave's A fragments (output block w)
  Raw ring[RES ? 1 : kRing];            // !RES: the next K-steps' fragments
  Raw dr[PD];                           // the next tile's dL/dout
  float h[L][RB][16];                   // h_l of this wave's 16 features of row n of each block (l >= 1)

  __device__ __forceinline__ bool owns(int l) const { return 32 * w < dimw<N>(p, l); }
  __device__ __forceinline__ static Raw load_raw(rsrc_t r, uint32_t byte) {
    Raw v;
#pragma unroll
    for (int i = 0; i < NT; ++i) v.v[i] = buf_load16<f32x4>(r, byte + 16 * i);
    return v;
  }
  __device__ __forceinline__ static Opnd to_op(const Raw& v) {
    if constexpr (EM == EM_F32) {
      const f32x4 a = v.v[0], b = v.v[NT - 1];
      const float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
      return make_op<EM>(f);
    } else {
      return Opnd{__builtin_bit_cast(f16x8, v.v[0]), f16x8{}};
    }
  }

  // Fragment (block w, K-step s) of layer l: lane (i, g) holds
  // W_l[outfeat(w, i)][16s + 8g + 0..7].  Rows and columns past the true
  // widths read zeros (offsets past the resource).
  template <int l>
  __device__ __forceinline__ Raw load_frag(int s) const {
    const int K = dimw<N>(p, l), Nout = dimw<N>(p, l + 1);
    if constexpr (PK) {  // (a wave past the layer's width, a K-step past the padded width: past the resource)
      const int KP = pack_ks(Nout);
      const rsrc_t r = make_rsrc(p.wp[l], (uint32_t)(pack_frags(K, Nout) * 1024));
      return load_raw(r, s < KP ? (uint32_t)((w * KP + s) * 64 + lane) * 16u : kPast);
    }
    const rsrc_t r = make_rsrc(p.w[l], (uint32_t)(K * Nout * kEs<EM>));
    const int c = 16 * s + 8 * g;
    const uint32_t off = (uint32_t)(outfeat(w, n) * Nout + c) * kEs<EM>;
    return load_raw(r, !N::gen || c < Nout ? off : kPast);
  }
  template <int l = G::LO>
  __device__ __forceinline__ void load_all_frags() {
    if constexpr (l < L) {
      if (owns(l)) {
#pragma unroll
        for (int s = 0; s < G::ks(l); ++s) fr[l][s] = to_op(load_frag<l>(s));
      }
      load_all_frags<l + 1>();
    }
  }
  template <int l>
  __device__ __forceinline__ void request() {
    if constexpr (!RES) {
#pragma unroll
      for (int t = 0; t < kRing; ++t) {
        ring[t] = load_frag<l>(t);
        __builtin_amdgcn_sched_barrier(0);  // in this order: the K loop counts them
      }
    }
  }

  // dL/dout of the tile at row0: piece q = tid + k * threads is row q / OCH,
  // elements 8 (q % OCH) .. + 7.  Row stride 0 broadcasts row 0; a negative one
  // (MLPMK_DOUT_SCALAR) one element to every row and feature below the output
  // width.  Rows past the batch and features past the width read zeros.
  __device__ __forceinline__ void load_dout(int64_t row0) {
    const int OW = dimw<N>(p, L);
    const int64_t st = p.dout_stride;
    const uint32_t nr = rows_at(p.M, row0, ROWS);
    const bool scalar = st < 0;
    const int64_t str = st > 0 ? st : 0;
    const uint32_t bytes = !nr ? 0u : scalar ? (uint32_t)kEs<EM> : (uint32_t)(((nr - 1) * str + OW) * kEs<EM>);
    const rsrc_t r = make_rsrc(static_cast<const char*>(p.dout) + row0 * str * kEs<EM>, bytes);
    const uint32_t past = bytes;  // (not kPast: rows of a wide gradient may lie more than 2 GiB apart)
#pragma unroll
    for (int k = 0; k < PD; ++k) {
      const int q = (int)threadIdx.x + k * G::NWV * 64, row = q / OCH, c = 8 * (q % OCH);
      const bool ok = (uint32_t)row < nr && c < OW;
      if (scalar) {
        if constexpr (EM == EM_F32) {
          const float v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, ok ? 0 : (int)past, 0, 0));
          dr[k].v[0] = dr[k].v[NT - 1] = f32x4{v, v, v, v};
        } else {
          const int v = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r, ok ? 0 : (int)past, 0, 0);
          const int vv = v | (v << 16);
          dr[k].v[0] = __builtin_bit_cast(f32x4, (i32x4){vv, vv, vv, vv});
        }
      } else {
        dr[k] = load_raw(r, ok ? (uint32_t)(row * str + c) * kEs<EM> : past);
      }
    }
  }
  __device__ __forceinline__ void commit_dout() {
#pragma unroll
    for (int k = 0; k < PD; ++k) {
      const int q = (int)threadIdx.x + k * G::NWV * 64, row = q / OCH, c = q % OCH;
      if (ROWS * OCH % (G::NWV * 64) != 0 && row >= ROWS) continue;
      const Opnd o = to_op(dr[k]);
      tile[par][0][slot<CH>(row, c)] = o.h;
      if constexpr (NT == 2) tile[par][NT - 1][slot<CH>(row, c)] = o.l;
    }
  }

  // h_l for this wave's 16 features of row n of each row block (features 32w +
  // 8g + [0..7] and 32w + 16 + 8g + [0..7]), fp32.  Past the batch the
  // resource is empty and the loads return zeros.
  template <int l>
  __device__ __forceinline__ void load_h(int64_t row0) {
    const int HW = dimw<N>(p, l);
    const rsrc_t r = make_rsrc(p.stash[l - 1] + row0 * HW, owns(l) ? rows_at(p.M, row0, ROWS) * HW * 4u : 0u);
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const uint32_t e = (uint32_t)((32 * b + n) * HW + 32 * w + 8 * g) * 4;
      const f32x4 v0 = buf_load16<f32x4>(r, e), v1 = buf_load16<f32x4>(r, e + 16);
      const f32x4 v2 = buf_load16<f32x4>(r, e + 64), v3 = buf_load16<f32x4>(r, e + 80);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h[l][b][j] = v0[j];
        h[l][b][4 + j] = v1[j];
        h[l][b][8 + j] = v2[j];
        h[l][b][12 + j] = v3[j];
      }
    }
  }
  template <int l = L - 1>
  __device__ __forceinline__ void load_all_h(int64_t row0) {
    if constexpr (l >= 1) {
      load_h<l>(row0);
      load_all_h<l - 1>(row0);
    }
  }

  // Stores 16 values of row 32b + n (features 32w + 8g + [0..7], 32w + 16 +
  // 8g + [0..7]) into a [M, W] tensor of the mode's element type; halves past
  // the true width are dropped.
  __device__ __forceinline__ void store_row16(rsrc_t r, int W, int b, const float (&v)[16]) const {
    const uint32_t e = (uint32_t)((32 * b + n) * W + 32 * w + 8 * g);
    if (!N::gen || 32 * w < W) store8<EM>(r, e, v);
    if (!N::gen || 32 * w + 16 < W) store8<EM>(r, e + 16, v + 8);
  }
  __device__ __forceinline__ rsrc_t rows_rsrc(void* base, int W, int64_t row0) const {
    return make_rsrc(static_cast<char*>(base) + row0 * W * kEs<EM>, rows_at(p.M, row0, ROWS) * W * kEs<EM>);
  }

  // The MFMAs of layer l: acc[b] = W_l rows [32w, + 32) . dz_l of row block b.
  template <int l>
  __device__ __forceinline__ void chain(f32x16 (&acc)[RB], int t) {
    const f16x8* th = tile[t][0];
    const f16x8* tl = tile[t][NT - 1];
    auto read = [&](Opnd (&o)[RB], int s) {
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        o[b].h = th[slot<CH>(32 * b + n, 2 * s + g)];
        o[b].l = NT == 2 ? tl[slot<CH>(32 * b + n, 2 * s + g)] : f16x8{};
      }
    };
    Opnd in[2][RB];
    read(in[0], 0);
    if constexpr (RES) {
#pragma unroll
      for (int s = 0; s < G::ks(l); ++s) {
        if (s + 1 < G::ks(l)) read(in[(s + 1) & 1], s + 1);
#pragma unroll
        for (int b = 0; b < RB; ++b) acc[b] = mma<EM>(fr[l][s], in[s & 1][b], acc[b]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // Whole turns of kRing K-steps: past the true width both the tile and the
      // fragments hold zeros up to a multiple of 64 features.  (Zero fragments
      // alone are not enough: an infinite dz would meet them as inf * 0 = NaN.)
      const int KS = pack_ks(dimw<N>(p, l + 1));
      for (int c = 0; c < KS; c += kRing) {
#pragma unroll
        for (int t = 0; t < kRing; ++t) {
          read(in[(t + 1) & 1], c + t + 1 < KS ? c + t + 1 : 0);  // (past the last one: K-step 0 again)
          const Opnd a = to_op(ring[t]);
#pragma unroll
          for (int b = 0; b < RB; ++b) acc[b] = mma<EM>(a, in[t & 1][b], acc[b]);
          ring[t] = load_frag<l>(c + kRing + t);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }

  // Layer l of the tile at row0 (the next one at `next`): tile[par] holds dz_l.
  // Owning waves compute their 32 features of dz_{l-1} = (dz_l W_l^T) *
  // sigma(h_l) (or of dx for l = 0), store them and hand them on.
  template <int l>
  __device__ __forceinline__ void layer(int64_t row0, int64_t next) {
    constexpr bool HAND = l >= 1 && l - 1 >= G::LO;  // another layer follows
    f32x16 acc[RB] = {};
    if (owns(l)) chain<l>(acc, par);
    request<(HAND ? l - 1 : L - 1)>();
    par ^= 1;
    if constexpr (l >= 1) {
      const int W = dimw<N>(p, l);
      const rsrc_t dz = rows_rsrc(p.dz[l - 1], W, row0);
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        float v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = acc[b][j] * sig_from_h(h[l][b][j]);
        store_row16(dz, W, b, v);  // for the weight-gradient pass
        if constexpr (HAND) {      // and for the next layer, through the tile
          if (!N::gen || 32 * w < ((W + 63) & ~63)) {
            Opnd lo = make_op<EM>(*reinterpret_cast<const float(*)[8]>(v));
            Opnd hi = make_op<EM>(*reinterpret_cast<const float(*)[8]>(v + 8));
            // (widths are multiples of 16: past them zeros, whatever the products were)
            if (N::gen && 32 * w >= W) lo = Opnd{f16x8{}, f16x8{}};
            if (N::gen && 32 * w + 16 >= W) hi = Opnd{f16x8{}, f16x8{}};
            tile[par][0][slot<CH>(32 * b + n, 4 * w + g)] = lo.h;
            tile[par][0][slot<CH>(32 * b + n, 4 * w + 2 + g)] = hi.h;
            if constexpr (NT == 2) {
              tile[par][NT - 1][slot<CH>(32 * b + n, 4 * w + g)] = lo.l;
              tile[par][NT - 1][slot<CH>(32 * b + n, 4 * w + 2 + g)] = hi.l;
            }
          }
        }
      }
      load_h<l>(next);
    } else {
      const int W = dimw<N>(p, 0);
      const rsrc_t dx = rows_rsrc(p.dx, W, row0);
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        float v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = acc[b][j];
        if (owns(0)) store_row16(dx, W, b, v);
      }
    }
    if constexpr (HAND) {
      // The whole of dz_{l-1} of these rows is in the tile.  (The other tile,
      // read just now, is written after this barrier at the earliest.)
      __syncthreads();
      layer<l - 1>(row0, next);
    }
  }
};

template <class N, int EM, bool DX, bool RES, int RB, bool PK>
__global__ __launch_bounds__((DgGeo<N, DX>::NWV * 64)) void tp_dgrad_kernel(TpParams p) {
  using G = DgGeo<N, DX>;
  using W = DgWave<N, EM, DX, RES, RB, PK>;
  static_assert(G::valid(), "two-pass backward shape");
  __shared__ f16x8 tile[2][W::NT][W::ROWS * G::CH];  // two exchange tiles (hi, and lo with fp32 tensors)
  const int lane = threadIdx.x & 63;
  W wv{p, tile, lane, lane & 31, lane >> 5, __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))};
  const int64_t ntiles = (p.M + W::ROWS - 1) / W::ROWS;
  if (p.zero_dw) {
    // Written (=) rather than accumulated dW: cleared here, before the
    // weight-gradient pass adds its tiles (the next launch on the stream).
    // Every layer's d[l] * d[l+1] is a multiple of 128 (widths multiples of
    // 16, the output width of 8) and dw is 16-byte aligned.
    const int64_t nthr = (int64_t)gridDim.x * blockDim.x;
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
#pragma unroll
    for (int l = 0; l < N::L; ++l) {
      const int64_t n4 = (int64_t)dimw<N>(p, l) * dimw<N>(p, l + 1) / 4;
      f32x4* const d = reinterpret_cast<f32x4*>(p.dw[l]);
      for (int64_t i = tid; i < n4; i += nthr) d[i] = f32x4{};
    }
  }
  int64_t t = blockIdx.x;
  wv.load_dout(t * W::ROWS);
  wv.template load_all_h<>(t * W::ROWS);  // (from HBM: the longest wait first)
  if constexpr (RES) wv.template load_all_frags<>();  // (L2 hits after the first workgroup)
  wv.template request<N::L - 1>();
  for (; t < ntiles; t += gridDim.x) {
    const int64_t row0 = t * W::ROWS, next = row0 + (int64_t)gridDim.x * W::ROWS;
    wv.commit_dout();
    wv.load_dout(next);
    __syncthreads();  // dL/dout of these rows is in the tile
    wv.template layer<N::L - 1>(row0, next);
  }
}

// ---------------------------------------------------------------------------
// Pass 2: weight gradients
// ---------------------------------------------------------------------------

// A workgroup owns TQI x TQO quads (64 x 64 blocks of dW_l): its LDS tile rows
// hold 64 TQI features of a_l and then 64 TQO features of dz_l, RP rows per
// pass.  With one quad its four waves own one 32 x 32 tile each; otherwise a
// wave owns a quad.  Every wave runs all the K-rows of a pass for its tiles.
// KG wave groups (each with its own LDS tile) take the chunk's passes in
// turns and add up through LDS at the end: the rows in flight of that many
// workgroups, for the atomics of one.
template <int EM, int TQI, int TQO, int KG>
struct WgGeo {
  static constexpr int QW = TQI * TQO;
  static constexpr int GW = QW == 1 ? 4 : QW;        // waves per group
  static constexpr int GT = 64 * GW, THREADS = KG * GT;
  static constexpr int TPW = QW == 1 ? 1 : 4;        // 32 x 32 tiles per wave
  static constexpr int FA = 64 * TQI, FZ = 64 * TQO, F = FA + FZ;
  static constexpr int NT = EM == EM_F32 ? 2 : 1;    // tiles: hi (and lo)
  static constexpr int RP = F > 256 ? 128 : 32768 / F / NT;  // rows per pass
  static constexpr int PA = RP * FA / 8 / GT;        // 8-element pieces of a_l per thread per pass
  static constexpr int PZ = RP * FZ / 8 / GT;        // and of dz_l
  static constexpr int KS = RP / 16;                 // K-steps per pass
  static constexpr int TILE = NT * RP * F;           // 16-bit elements of a group's tiles
  static constexpr int LDS_BYTES = KG * TILE * 2;
  static_assert(QW == 1 || QW == 4 || (QW == 8 && EM != EM_F32), "one quad per workgroup or one per wave");
  static_assert(KG == 1 || (KG == 2 && QW == 4 && LDS_BYTES >= 2 * GW * 2 * 4096), "the groups' sums meet in the tiles");
};

// Tile layout: element (r, f) of a tile with F features per row sits at
// r*F + (f ^ swz(r, F)), where F is a power of two (else each half of the row
// for itself); the XOR moves whole 8-feature chunks, so 16-byte
// writes and 8-byte transposed reads stay contiguous, and the four rows of
// one transposed read land in four distinct 16-feature windows.
__device__ __forceinline__ int swz(int r, int F) {
  return (16 * (r & 3) + 8 * ((r >> 2) & 1) + 64 * ((r >> 3) & 1)) & (F - 1);
}

// MFMA operand for features fb .. fb+31 over rows 16kk .. 16kk+15 of a tile of
// F features a row (F0, FS: first feature and extent of the XOR):
// lane (m, g) gets rows 16kk + 8g + [0..7] of feature fb + m, through two
// transposing reads (per 16-lane group: result lane i, element j is element
// i & 3 of the 8 bytes addressed by lane (i >> 2) + 4j).
template <int F, int F0, int FS>
__device__ __forceinline__ f16x8 xread(const f16* t, int fb, int kk, const int (&rrow)[2], int rcol) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  s16x4 h[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int r = rrow[k];
    const f16* a = t + (16 * kk + r) * F + F0 + ((fb + rcol) ^ swz(r, FS));
    h[k] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)const_cast<f16*>(a));
  }
  return __builtin_bit_cast(f16x8, __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3, 4, 5, 6, 7));
}

// Where a workgroup's operands come from: a_l (x for l = 0, else the fp32
// stash) and dz_l (dL/dout for the last layer, else the workspace).
struct WgSrc {
  const char* base;  // element 0 of the first row of the chunk
  int64_t stride;    // elements between rows; 0 = one row for all; -1 = one element for all
  int es;            // 2 (16-bit) or 4 (fp32)
  int width;         // true features
  int f0;            // first feature of the workgroup's block
  uint32_t bytes;    // resource size from base
};

// MINW: waves per SIMD the register allocation must leave room for: 2 for the
// 4-wave kernels when the grid has more workgroups than CUs (two workgroups
// per CU keep twice the rows in flight).
template <class N, int EM, int TQI, int TQO, int KG, int MINW>
__global__ __launch_bounds__((WgGeo<EM, TQI, TQO, KG>::THREADS), MINW) void tp_wgrad_kernel(TpParams p) {
  using G = WgGeo<EM, TQI, TQO, KG>;
  constexpr int F = G::F, RP = G::RP, NT = G::NT, GT = G::GT;
  constexpr bool kPow2 = (F & (F - 1)) == 0;
  __shared__ __attribute__((aligned(16))) char smem[G::LDS_BYTES];
  const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / GT);  // this wave's group
  f16* const tiles = reinterpret_cast<f16*>(smem) + kg * G::TILE;
  const int L = N::L;
  // Task: (layer, quad block) from blockIdx.y, row chunk from blockIdx.x.
  int l = 0, bi = 0, bo = 0;
  {
    int t = blockIdx.y;
    for (int i = 0; i < L; ++i) {
      const int ni = (dimw<N>(p, i) + G::FA - 1) / G::FA, no = (dimw<N>(p, i + 1) + G::FZ - 1) / G::FZ;
      if (t < ni * no) {
        l = i;
        bi = t / no;
        bo = t % no;
        break;
      }
      t -= ni * no;
    }
  }
  const int K = dimw<N>(p, l), NO = dimw<N>(p, l + 1);
  const int64_t passes = (p.M + RP - 1) / RP;  // split evenly over the chunks
  const int64_t r_begin = passes * blockIdx.x / gridDim.x * RP;
  const int64_t r_next = passes * (blockIdx.x + 1) / gridDim.x * RP;
  const int64_t r_end = r_next < p.M ? r_next : p.M;
  const int64_t nrows = r_end - r_begin;
  // Sources.  Resources clip to the chunk's rows, so loads past them read 0.
  WgSrc sa, sz;
  {
    const bool x = l == 0;
    sa.es = x ? kEs<EM> : 4;
    sa.stride = K;
    sa.width = K;
    sa.f0 = G::FA * bi;
    sa.base = x ? static_cast<const char*>(p.x) + r_begin * K * kEs<EM>
                : reinterpret_cast<const char*>(p.stash[l - 1] + r_begin * K);
    sa.bytes = (uint32_t)(nrows * K * sa.es);
    const bool top = l == L - 1;
    sz.es = kEs<EM>;
    sz.width = NO;
    sz.f0 = G::FZ * bo;
    if (top) {
      sz.stride = p.dout_stride < 0 ? -1 : p.dout_stride;
      const int64_t st = sz.stride > 0 ? sz.stride : 0;
      sz.base = static_cast<const char*>(p.dout) + r_begin * st * kEs<EM>;
      sz.bytes = sz.stride < 0 ? (uint32_t)kEs<EM> : (uint32_t)(((nrows - 1) * st + NO) * kEs<EM>);
    } else {
      sz.stride = NO;
      sz.base = static_cast<const char*>(p.dz[l]) + r_begin * NO * kEs<EM>;
      sz.bytes = (uint32_t)(nrows * NO * kEs<EM>);
    }
  }
  const rsrc_t ra = make_rsrc(sa.base, sa.bytes), rz = make_rsrc(sz.base, sz.bytes);
  const int tid = (int)threadIdx.x - kg * GT, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

  // Loads of one pass.  a_l pieces first (8 features each), then dz_l
  // pieces: piece k of this thread is q = tid + GT k, row q / (FA / 8)
  // (resp. FZ / 8), chunk q % (FA / 8) -- consecutive threads read
  // consecutive 16-byte pieces of a row.  Raw payloads: up to 32 bytes (8
  // fp32) per piece, kept until the tile is free (16-bit dz: 16 bytes).
  struct Raw {
    f32x4 a, b;
  };
  struct Raw16 {
    f32x4 a;
  };
  Raw raw_a[G::PA];
  typename std::conditional<EM == EM_F32, Raw, Raw16>::type raw_z[G::PZ];
  auto issue_src = [&](auto& raw, const WgSrc& s, rsrc_t rr, int FS, int64_t prow) {
    constexpr int NP = sizeof(raw) / sizeof(raw[0]);
    constexpr bool WIDE = sizeof(raw[0]) > 16;  // the piece may be fp32
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int q = tid + GT * k, r = q / (FS / 8), c = q % (FS / 8);
      const int f = s.f0 + 8 * c;
      const int64_t row = prow + r;
      const bool ok = f < s.width && row < nrows;
      const int64_t e = s.stride < 0 ? 0 : row * s.stride + f;
      raw[k].a = f32x4{};
      if constexpr (WIDE) raw[k].b = f32x4{};
      if (!ok) continue;
      if (WIDE && s.es == 4) {
        raw[k].a = buf_load16<f32x4>(rr, (uint32_t)(e * 4));
        if constexpr (WIDE) raw[k].b = buf_load16<f32x4>(rr, (uint32_t)(e * 4 + 16));
      } else if (s.stride < 0) {  // one 16-bit element for every row and feature
        const int v = __builtin_amdgcn_raw_buffer_load_b16(rr, 0, 0, 0);
        const int vv = (v & 0xffff) | (v << 16);
        raw[k].a = __builtin_bit_cast(f32x4, (i32x4){vv, vv, vv, vv});
      } else {
        raw[k].a = buf_load16<f32x4>(rr, (uint32_t)(e * 2));
      }
    }
  };
  auto issue = [&](int64_t prow) {  // rows prow .. prow + RP - 1 of the chunk
    issue_src(raw_a, sa, ra, G::FA, prow);
    issue_src(raw_z, sz, rz, G::FZ, prow);
  };
  // Convert a pass's pieces and write them into the tile(s): a_l at
  // features [0, FA), dz_l at [FA, F) of each tile row.
  auto commit_src = [&](const auto& raw, const WgSrc& s, int FS, int fbase) {
    constexpr int NP = sizeof(raw) / sizeof(raw[0]);
    constexpr bool WIDE = sizeof(raw[0]) > 16;
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int q = tid + GT * k, r = q / (FS / 8), c = q % (FS / 8);
      Opnd o;
      o.h = __builtin_bit_cast(f16x8, raw[k].a);
      o.l = f16x8{};
      if constexpr (WIDE) {
        if (s.es == 4) {
          float v[8] = {raw[k].a[0], raw[k].a[1], raw[k].a[2], raw[k].a[3],
                        raw[k].b[0], raw[k].b[1], raw[k].b[2], raw[k].b[3]};
          if (s.stride < 0) {  // (fp32 scalar: element 0 everywhere)
#pragma unroll
            for (int j = 1; j < 8; ++j) v[j] = v[0];
          }
          o = make_op<EM>(v);
        }
      }
      const int off = r * F + (kPow2 ? (fbase + 8 * c) ^ swz(r, F) : fbase + ((8 * c) ^ swz(r, FS)));
      *reinterpret_cast<f16x8*>(tiles + off) = o.h;
      if constexpr (NT == 2) *reinterpret_cast<f16x8*>(tiles + RP * F + off) = o.l;
    }
  };
  auto commit = [&]() {
    commit_src(raw_a, sa, G::FA, 0);
    commit_src(raw_z, sz, G::FZ, G::FA);
  };

  // Wave w: with one quad, tile (w >> 1, w & 1) of it; with four, quad
  // (w / TQO, w % TQO).
  const int qi = G::QW == 1 ? 0 : w / TQO, qo = G::QW == 1 ? 0 : w % TQO;
  int rrow[2], rcol;
  {
    const int q = lane >> 4, i = lane & 15;
    rrow[0] = 8 * (q >> 1) + (i >> 2);
    rrow[1] = rrow[0] + 4;
    rcol = 16 * (q & 1) + 4 * (i & 3);
  }
  f32x16 acc[G::TPW] = {};
  auto opnd_a = [&](int fb, int kk) {
    constexpr int FS = kPow2 ? F : G::FA;
    Opnd o;
    o.h = xread<F, 0, FS>(tiles, fb, kk, rrow, rcol);
    o.l = NT == 2 ? xread<F, 0, FS>(tiles + RP * F, fb, kk, rrow, rcol) : f16x8{};
    return o;
  };
  auto opnd_z = [&](int fb, int kk) {
    constexpr int F0 = kPow2 ? 0 : G::FA, FS = kPow2 ? F : G::FZ;
    Opnd o;
    o.h = xread<F, F0, FS>(tiles, (kPow2 ? G::FA : 0) + fb, kk, rrow, rcol);
    o.l = NT == 2 ? xread<F, F0, FS>(tiles + RP * F, (kPow2 ? G::FA : 0) + fb, kk, rrow, rcol) : f16x8{};
    return o;
  };
  const int npass = (int)((nrows + RP - 1) / RP);
  // (A group's turn past the last pass reads nothing and adds zeros: every
  // wave runs the same barriers.)
  issue((int64_t)kg * RP);
  for (int ps = kg; ps - kg < npass; ps += KG) {
    __syncthreads();  // the previous pass's reads are done
    commit();
    if (ps - kg + KG < npass) issue((int64_t)(ps + KG) * RP);
    __syncthreads();  // the tile is written
    // (K-steps past the chunk's last row read zeros: the loads were masked.)
#pragma unroll
    for (int kk = 0; kk < G::KS; ++kk) {
      if constexpr (G::QW == 1) {
        acc[0] = mma<EM>(opnd_a(32 * (w >> 1), kk), opnd_z(32 * (w & 1), kk), acc[0]);
      } else {
        const Opnd a0 = opnd_a(64 * qi, kk), a1 = opnd_a(64 * qi + 32, kk);
        const Opnd b0 = opnd_z(64 * qo, kk), b1 = opnd_z(64 * qo + 32, kk);
        acc[0] = mma<EM>(a0, b0, acc[0]);
        acc[1] = mma<EM>(a0, b1, acc[1]);
        acc[2] = mma<EM>(a1, b0, acc[2]);
        acc[3] = mma<EM>(a1, b1, acc[3]);
      }
    }
  }
  if constexpr (KG == 2) {
    // Group 0 takes tiles 0 and 1 of every quad, group 1 tiles 2 and 3: each
    // leaves the other's two in LDS.
    float* const sum = reinterpret_cast<float*>(smem) + w * 2048 + lane;
    __syncthreads();  // the last pass's reads are done
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) sum[kg * G::GW * 2048 + t * 1024 + e * 64] = kg ? acc[t][e] : acc[2 + t][e];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float v = sum[(1 - kg) * G::GW * 2048 + t * 1024 + e * 64];
        acc[t][e] = (kg ? acc[2 + t][e] : acc[t][e]) + v;
      }
  }

  // Output: tile t = 2 ti + to of quad (qi, qo): C lane (o, g), register e
  // holds dW_l[i][o] for i = 8 (e >> 2) + 4 g + (e & 3) within the tile;
  // added to dw with fp32 atomics.
  auto write_tile = [&](const f32x16& a, int t) {
    const int ti = t >> 1, to = t & 1;
    const int i0 = G::FA * bi + 64 * qi + 32 * ti, o = G::FZ * bo + 64 * qo + 32 * to + (lane & 31);
    const int g = lane >> 5;
    float* const dst = p.dw[l];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int i = i0 + 8 * (e >> 2) + 4 * g + (e & 3);
      if (i < K && o < NO) unsafeAtomicAdd(dst + (int64_t)i * NO + o, a[e]);
    }
  };
  if constexpr (G::QW == 1) {
    write_tile(acc[0], w);
  } else if constexpr (KG == 2) {
#pragma unroll
    for (int t = 0; t < 2; ++t) write_tile(acc[t], 2 * kg + t);
  } else {
#pragma unroll
    for (int t = 0; t < 4; ++t) write_tile(acc[t], t);
  }
}

}  // namespace tp

// ---------------------------------------------------------------------------
// Host dispatch
// ---------------------------------------------------------------------------

namespace {

// Per-device occupancy of one kernel (benign race: the value is idempotent).
int cached_occupancy(const void* kern, int threads, int* occ_out) {
  constexpr int kMaxDev = 64;
  struct Entry {
    const void* k;
    int occ;
  };
  static Entry cache[kMaxDev][96];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev >= 0 && dev < kMaxDev) {
    for (auto& c : cache[dev]) {
      if (c.k == kern && c.occ > 0) {
        *occ_out = c.occ;
        return MLPMK_OK;
      }
      if (!c.k) break;
    }
  }
  int occ = 0;
  int rc = kernel_occupancy(kern, threads, &occ);
  if (rc != MLPMK_OK) return rc;
  if (dev >= 0 && dev < kMaxDev) {
    for (auto& c : cache[dev])
      if (!c.k || c.k == kern) {
        c.occ = occ;
        c.k = kern;
        break;
      }
  }
  *occ_out = occ;
  return MLPMK_OK;
}

template <class N, int EM, bool DX, bool RES, int RB, bool PK = false>
int launch_dgrad_rb(const TpParams& p, int cus, hipStream_t st) {
  using G = tp::DgGeo<N, DX>;
  const void* kern = reinterpret_cast<const void*>(&tp::tp_dgrad_kernel<N, EM, DX, RES, RB, PK>);
  int occ = 0;
  int rc = cached_occupancy(kern, G::NWV * 64, &occ);
  if (rc != MLPMK_OK) return rc;
  const int64_t ntiles = (p.M + 32 * RB - 1) / (32 * RB);
  const int64_t cap = (int64_t)cus * occ;
  const int grid = (int)(ntiles < cap ? ntiles : cap);
  (void)hipGetLastError();
  hipLaunchKernelGGL((tp::tp_dgrad_kernel<N, EM, DX, RES, RB, PK>), dim3(grid), dim3(G::NWV * 64), 0, st, p);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? MLPMK_OK : hip_fail(e, "two-pass dgrad kernel launch");
}

// Tiles of 64 rows read the weights once for twice the rows, but hand a CU its
// rows in twice as large steps: at 20,000 rows two of them (128 rows) where
// tiles of 32 make three (96).  So 64 rows from 64 rows per CU on where that is
// at most 7 % more rows for the CU with most, or where the weights weigh more: hidden
// widths of 128 with fp32 tensors, of 192 and more in 16 bits.  With resident
// weights (RES) nothing is read again, and 64 rows pay from 512 per CU on.
// Whole backward, us, tiles of 64 / 32 rows: 3x128 fp32 20,000 rows 47 / 43,
// 65,536 85 / 83, 131,072 155 / 160, 600,000 642 / 667; 32-96-96-96-16 fp32 24,000
// 49 / 45, 131,072 175 / 192, 200,003 278 / 301; 5x128 fp32 24,000 85 / 87, 32,768 87 / 98;
// 16-144-144-144-144-72 bf16 20,000 with dx 88 / 75; 256-256-256-256 fp16 20,000
// 86 / 90; 4x160 fp16 17,000 66 / 64, 28,000 68 / 72.
template <int EM, bool RES>
bool dgrad_wide_tiles(const TpParams& p, int L, int cus) {
  if (RES) return p.M >= (int64_t)512 * cus;
  if (p.M <= (int64_t)64 * cus) return false;
  int hidden = p.dims[1];
  for (int l = 2; l < L; ++l) hidden = p.dims[l] < hidden ? p.dims[l] : hidden;
  if (hidden >= (EM == tp::EM_F32 ? 128 : 192)) return true;
  auto rounds = [&](int64_t rows) { return ((p.M + rows - 1) / rows + cus - 1) / cus; };
  return 200 * rounds(64) <= 107 * rounds(32);
}

template <class N, int EM, bool DX, bool RES>
int launch_dgrad(const TpParams& p, int cus, hipStream_t st) {
  if constexpr (EM != tp::EM_F32 && !RES) {
    if (p.wp[0]) return launch_dgrad_rb<N, EM, DX, RES, 2, true>(p, cus, st);
  }
  return dgrad_wide_tiles<EM, RES>(p, N::L, cus) ? launch_dgrad_rb<N, EM, DX, RES, 2>(p, cus, st)
                                                 : launch_dgrad_rb<N, EM, DX, RES, 1>(p, cus, st);
}

// Weight-gradient tiling (WgGeo): WG_QUAD, one 64 x 64 block per 4-wave
// workgroup, gives small batches enough workgroups; the others read each a_l
// and dz_l element fewer times.  WG_PAIR: 128 x 128 blocks, 8 waves in two
// groups (widths up to 128: each operand read once).  WG_WIDE: 128 x 256
// blocks, 8 waves (16-bit tensors of widths above 128: the fp32 activations
// read once, dz twice).
//
// The other forms win once the rows times the 64 x 64 blocks, each of which
// reads its rows again, reach a number that depends on the chunks S of
// WG_QUAD: where S is a multiple of the 8 XCDs, the blocks of a chunk run on
// one XCD and share its rows in that L2, and WG_QUAD holds out 2.5 times as
// long.  Whole backward, us, QUAD / WIDE (16-bit tensors; blocks, S):
// 256-256-256-256 [48, 10] 12,288 rows 62 / 63, 24,000 98 / 82; 6 x 256 [80, 6]
// 8,192 68 / 65, 24,000 172 / 123; 160-192-192-192-64 [30, 17] 12,288 43 / 51,
// 20,000 72 / 65; 256-256-8 [20, 25] 24,000 39 / 47, 40,000 59 / 58; but
// 128-256-256-128 [32, 16] 40,000 83 / 88, 50,000 103 / 99; 64-256-64 [8, 64]
// 100,003 78 / 84.  QUAD / PAIR (fp32 tensors, widths above 64: a block of 128 x
// 128 is mostly empty below): 3x128 [12, 42] 32,768 60 / 58, 65,536 100 / 85;
// 80-80-8 [6, 85] 40,000 34 / 36, 65,536 44 / 43; but 2x128 [8, 64] 80,000 69 /
// 74, 131,072 103.5 / 102; 4x128 [16, 32] 49,152 92 / 95, 80,000 154 / 147;
// 64-128-64 [4, 128] 200,003 112 / 123.
// 16-bit networks up to 128 wide keep WG_QUAD: they come here up to 16,384 rows
// only (bwd_path), so WG_PAIR is built for fp32 tensors and WG_WIDE for the
// runtime-width networks of 16-bit ones.
enum { WG_QUAD, WG_PAIR, WG_WIDE };

int quad_blocks(int L, const int* dims, int form) {
  const int fa = form == WG_QUAD ? 64 : 128, fz = form == WG_QUAD ? 64 : form == WG_PAIR ? 128 : 256;
  int n = 0;
  for (int l = 0; l < L; ++l) n += ((dims[l] + fa - 1) / fa) * ((dims[l + 1] + fz - 1) / fz);
  return n;
}

constexpr int64_t kPairMinRows = 32768;
int wgrad_form(int L, const int* dims, int64_t M, bool f32, int cus) {
  int wmax = 0;
  for (int i = 0; i <= L; ++i) wmax = dims[i] > wmax ? dims[i] : wmax;
  const int quads = quad_blocks(L, dims, WG_QUAD);
  const bool shared = 2 * cus >= quads && 2 * cus / quads % 8 == 0;
  if (wmax > 128) return M * quads >= (shared ? 1440000 : 540000) ? WG_WIDE : WG_QUAD;
  return f32 && wmax > 64 && M >= kPairMinRows && M * quads >= (shared ? 880000 : 360000) ? WG_PAIR : WG_QUAD;
}

// Longest row chunk with fp32 tensors.  A chunk's products of split
// operands accumulate in one MFMA chain per tile, three MFMAs per K-step, and
// over long chains that sum drifts: the last layer's dW of a 40,000,037-row
// batch (broadcast dout, so its exact value is a column sum) was off by
// 1.6e-4 with chunks of 234 K rows and 6.9e-5 with chunks of 117 K rows;
// the 16-bit one-pass kernel, one MFMA per K-step, stays at 1.6e-6 over
// 156 K rows per workgroup.  Past this length the pass takes more chunks
// (more atomics) instead.
constexpr int64_t kF32MaxChunkRows = 8192;

// Row chunks of the weight-gradient pass: as many as let every workgroup run
// at once (two 4-wave workgroups per CU, one of 8 waves; one more would run
// after the others), each a whole number of passes -- the fewest chunks that
// keep the longest one as short while chunks are a few passes long, else that
// many chunks with the passes spread evenly -- and with fp32 tensors of at
// most kF32MaxChunkRows rows.
int wgrad_chunks(int L, const int* dims, int64_t M, bool f32, int cus) {
  const int form = wgrad_form(L, dims, M, f32, cus);
  const int rp = (form == WG_QUAD ? 256 : 128) / (f32 ? 2 : 1);  // rows per pass (WgGeo::RP)
  const int nqb = quad_blocks(L, dims, form);
  const int64_t passes = (M + rp - 1) / rp;
  int64_t S = (int64_t)(form == WG_QUAD ? 2 : 1) * cus / nqb;
  if (S < 1) S = 1;
  const int64_t longest = (passes + S - 1) / S;
  if (longest < 4) S = (passes + longest - 1) / longest;
  if (f32 && S * (kF32MaxChunkRows / rp) < passes) S = (passes + kF32MaxChunkRows / rp - 1) / (kF32MaxChunkRows / rp);
  return (int)S;
}

template <class N, int EM, int TQI, int TQO, int KG, int MINW>
int launch_wgrad(const TpParams& p, int S, int nqb, hipStream_t st) {
  (void)hipGetLastError();
  hipLaunchKernelGGL((tp::tp_wgrad_kernel<N, EM, TQI, TQO, KG, MINW>), dim3(S, nqb),
                     dim3(tp::WgGeo<EM, TQI, TQO, KG>::THREADS), 0, st, p);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? MLPMK_OK : hip_fail(e, "two-pass wgrad kernel launch");
}

template <class N, int EM>
int launch_wgrad_form(const TpParams& p, int form, int S, int nqb, int cus, hipStream_t st) {
  if constexpr (EM == tp::EM_F32) {
    if (form == WG_PAIR) return launch_wgrad<N, EM, 2, 2, 2, 1>(p, S, nqb, st);
  } else if constexpr (N::gen) {
    if (form == WG_WIDE) return launch_wgrad<N, EM, 2, 4, 1, 1>(p, S, nqb, st);
  }
  return (int64_t)S * nqb > cus ? launch_wgrad<N, EM, 1, 1, 1, 2>(p, S, nqb, st)
                                : launch_wgrad<N, EM, 1, 1, 1, 1>(p, S, nqb, st);
}

int64_t round256(int64_t b) { return (b + 255) / 256 * 256; }

typedef Net<128, 128, 128, 128> TNet3L128;
template <int L>
struct GenTp;  // runtime widths up to 256 (16-bit tensors) / 128 (fp32)
template <>
struct GenTp<2> {
  typedef Gen<Net<256, 256, 256>> W;
  typedef Gen<Net<128, 128, 128>> F;
};
template <>
struct GenTp<3> {
  typedef Gen<Net<256, 256, 256, 256>> W;
  typedef Gen<Net<128, 128, 128, 128>> F;
};
template <>
struct GenTp<4> {
  typedef Gen<Net<256, 256, 256, 256, 256>> W;
  typedef Gen<Net<128, 128, 128, 128, 128>> F;
};
template <>
struct GenTp<5> {
  typedef Gen<Net<256, 256, 256, 256, 256, 256>> W;
  typedef Gen<Net<128, 128, 128, 128, 128, 128>> F;
};

bool is_3l128(int L, const int* dims) {
  return L == 3 && dims[0] == 128 && dims[1] == 128 && dims[2] == 128 && dims[3] == 128;
}

template <int EM, int L>
int dispatch_l(const TpParams& p, const int* dims, int S, hipStream_t st) {
  int cus = 0;
  int rc = current_device_cus(&cus);
  if (rc != MLPMK_OK) return rc;
  const bool dx = p.dx != nullptr;
  // Pass 1.
  if (L == 3 && is_3l128(L, dims)) {
    rc = dx ? launch_dgrad<TNet3L128, EM, true, true>(p, cus, st) : launch_dgrad<TNet3L128, EM, false, true>(p, cus, st);
  } else if constexpr (EM == tp::EM_F32) {
    typedef typename GenTp<L>::F NG;
    rc = dx ? launch_dgrad<NG, EM, true, false>(p, cus, st) : launch_dgrad<NG, EM, false, false>(p, cus, st);
  } else {
    typedef typename GenTp<L>::W NG;
    rc = dx ? launch_dgrad<NG, EM, true, false>(p, cus, st) : launch_dgrad<NG, EM, false, false>(p, cus, st);
  }
  if (rc != MLPMK_OK) return rc;
  // Pass 2 (the kernel reads only N's layer count and whether its widths are
  // fixed: one runtime-width instance per depth serves every shape).
  const int form = wgrad_form(L, dims, p.M, EM == tp::EM_F32, cus);
  const int nqb = quad_blocks(L, dims, form);
  typedef typename GenTp<L>::W NW;
  rc = L == 3 && is_3l128(L, dims) ? launch_wgrad_form<TNet3L128, EM>(p, form, S, nqb, cus, st)
                                   : launch_wgrad_form<NW, EM>(p, form, S, nqb, cus, st);
  return rc;
}

}  // namespace

// Shapes of the two-pass backward: 2..5 layers, input and hidden widths
// multiples of 16 and the output width a multiple of 8, all in [16, 256]
// for 16-bit tensors ([16, 128] for fp32 tensors).
bool tp_supported(int L, const int* dims, int dtype) {
  if (L < 2 || L > 5) return false;
  const int wmax = dtype == MLPMK_DTYPE_F32 ? 128 : 256;
  for (int i = 0; i < L; ++i)
    if (dims[i] < 16 || dims[i] > wmax || dims[i] % 16 != 0) return false;
  return dims[L] >= 8 && dims[L] <= wmax && dims[L] % 8 == 0;
}

// The packed weights' bytes, 0 where the pass takes them from W_l: fp32 tensors
// (split when loaded), widths up to 128, and batches up to this many rows,
// where the packing launch (4 us) costs more than it saves.
constexpr int64_t kPackMinRows = 32768;
int64_t tp_pack_bytes(int L, const int* dims, int dtype, int64_t M) {
  int wmax = 0;
  int64_t b = 0;
  for (int l = 0; l < L; ++l) {
    b += (int64_t)tp::pack_frags(dims[l], dims[l + 1]) * 1024;
    wmax = dims[l] > wmax ? dims[l] : wmax;
  }
  wmax = dims[L] > wmax ? dims[L] : wmax;
  return dtype != MLPMK_DTYPE_F32 && wmax > 128 && M >= kPackMinRows ? b : 0;
}

// Workspace of the two-pass backward: dz_0 .. dz_{L-2} ([M, d[l+1]] each,
// 16-bit or fp32 elements, 256-byte aligned), then the packed weights.
int tp_workspace_bytes(int L, const int* dims, int dtype, int64_t M, int64_t* bytes) {
  const int es = dtype == MLPMK_DTYPE_F32 ? 4 : 2;
  int64_t b = tp_pack_bytes(L, dims, dtype, M);
  for (int l = 0; l + 1 < L; ++l) b += round256(M * dims[l + 1] * es);
  *bytes = b;
  return MLPMK_OK;
}

// The two-pass backward.  bp carries the tensors as bwd_common validated
// them; ws holds at least tp_workspace_bytes.
int tp_dispatch(int L, const int* dims, int dtype, const BwdParams& bp, void* ws, hipStream_t st) {
  int cus = 0;
  int rc = current_device_cus(&cus);
  if (rc != MLPMK_OK) return rc;
  TpParams p = {};
  p.x = bp.x;
  for (int l = 0; l < L; ++l) {
    p.w[l] = bp.w[l];
    p.dw[l] = bp.dw[l];
  }
  for (int l = 0; l + 1 < L; ++l) p.stash[l] = bp.stash[l];
  p.dout = bp.dout;
  p.dout_stride = bp.dout_stride;
  p.dx = bp.dx;
  p.M = bp.M;
  p.zero_dw = bp.write_dw;
  for (int l = 0; l <= L; ++l) p.dims[l] = dims[l];
  const int es = dtype == MLPMK_DTYPE_F32 ? 4 : 2;
  char* c = static_cast<char*>(ws);
  for (int l = 0; l + 1 < L; ++l) {
    p.dz[l] = c;
    c += round256(bp.M * dims[l + 1] * es);
  }
  if (bp.pack_room && tp_pack_bytes(L, dims, dtype, bp.M) > 0) {
    tp::PackParams pk = {};
    pk.L = L;
    for (int l = 0; l < L; ++l) {
      pk.w[l] = bp.w[l];
      p.wp[l] = pk.dst[l] = reinterpret_cast<f16*>(c);
      const int frags = tp::pack_frags(dims[l], dims[l + 1]);
      pk.first[l + 1] = pk.first[l] + frags * 64;
      c += (int64_t)frags * 1024;
    }
    for (int l = 0; l <= L; ++l) pk.dims[l] = dims[l];
    (void)hipGetLastError();
    hipLaunchKernelGGL(tp::tp_pack_kernel, dim3((pk.first[L] + 255) / 256), dim3(256), 0, st, pk);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, "weight packing kernel launch");
  }
  const int S = wgrad_chunks(L, dims, bp.M, dtype == MLPMK_DTYPE_F32, cus);
  const int em = dtype == MLPMK_DTYPE_F32 ? tp::EM_F32 : dtype == MLPMK_DTYPE_BF16 ? tp::EM_BF16 : tp::EM_F16;
  switch (em * 8 + L) {
#define MLPMK_TP_CASE(E, LL) \
  case E * 8 + LL: return dispatch_l<E, LL>(p, dims, S, st);
    MLPMK_TP_CASE(tp::EM_F16, 2) MLPMK_TP_CASE(tp::EM_F16, 3) MLPMK_TP_CASE(tp::EM_F16, 4) MLPMK_TP_CASE(tp::EM_F16, 5)
    MLPMK_TP_CASE(tp::EM_BF16, 2) MLPMK_TP_CASE(tp::EM_BF16, 3) MLPMK_TP_CASE(tp::EM_BF16, 4)
    MLPMK_TP_CASE(tp::EM_BF16, 5) MLPMK_TP_CASE(tp::EM_F32, 2) MLPMK_TP_CASE(tp::EM_F32, 3)
    MLPMK_TP_CASE(tp::EM_F32, 4) MLPMK_TP_CASE(tp::EM_F32, 5)
#undef MLPMK_TP_CASE
    default: return fail(MLPMK_ERR_UNSUPPORTED_SHAPE, "two-pass backward: %d layers", L);
  }
}

}  // namespace mlpmk
