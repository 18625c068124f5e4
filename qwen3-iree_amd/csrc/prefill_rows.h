// Products of a short prompt's layer (up to 128 tokens), each
// workgroup holding the whole K of its few weight rows ("row products"),
// included by prefill_kernels.hip.
//
// A short prompt's layer is bound by launches and load latency, not by bytes
// or MFMAs: 31 MB of f16 weights take 6 us at 5 TB/s, while eleven launches
// whose workgroups walk K stage by stage took 43-51 us for 1-128 tokens.  So
// each of these kernels asks for everything it will multiply at once (no
// stage waits for another's load), and does the work of the launches around
// it under that latency: rms_norm of the token rows in the prologue; head
// norms, RoPE and the cache writes in the q/k/v epilogue; the K ranges of one
// output summed through LDS instead of a second launch, with the residual
// add.  Measured per layer (f16 weights, 1 / 24 / 33 / 64 / 128 tokens):
// 42.6 / 46.6 / 50.1 / 51.2 / 50.6 us with the tiled GEMMs, 26.7 / 28.9 / 33.0
// / 33.7 / 39.9 us with these; over the Q8_0 stacks 43.1 / 46.7 / 49.7 / 50.1 /
// 52.9 and 26.4 / 29.3 / 33.9 / 34.3 / 41.3 us.
//
// Every output is a sum of chains of v_mfma_f32_16x16x32_f16 in K order, the
// chains added in order in f32: q/k/v and gate/up eight chains of 128 k (q/k/v
// with RoPE one of 1024), attn_o and ffn_down chains of 256 k as the tiled
// split-K GEMMs have them.  The chains depend on the number of tokens only, so
// both weight forms give the same bits.  Norms, RoPE and epilogues are the
// device functions every other kernel uses.
#ifndef QWEN3_PREFILL_ROWS_H
#define QWEN3_PREFILL_ROWS_H

namespace {

// A wave's 16 weight rows over K k, on their way from memory to MFMA operands.
// Loads are contiguous along the rows (a load whose lanes gather 64 bytes from
// each of 16 rows takes the vector memory path 65-100 cycles against 16), so a
// lane does not receive the operand it needs: a stage is written to the wave's
// own LDS slot and read back as fragments.  LDS operations of one wave
// complete in order, so the slot needs no barrier and one slot serves every
// stage.
//
// f16: a stage is 128 k, 4 loads of 4 rows x 256 bytes; row r's 16-byte chunk
// c sits in slot c ^ r of its 256 bytes.
// Q8_0: a stage is 256 k (8 blocks), 272 bytes of each row as in memory in
// 16-byte pieces, or with K = 128 its 136 bytes in 8-byte pieces; five loads of
// which the last repeats piece 271.
template <bool Q8, int K>
struct WRows {
  static constexpr int kStageK = Q8 && K >= 256 ? 256 : 128;
  static constexpr int kPiece = Q8 && K < 256 ? 8 : 16;  // bytes per lane and load
  static constexpr int kQRow = 34 * kStageK / 32;
  static constexpr int kStages = K / kStageK;
  static constexpr int kLoads = Q8 ? 5 : 4;      // per lane and stage
  static constexpr int kSlot = Q8 ? 5 * 64 * kPiece : 4096;
  typedef uint32_t Piece __attribute__((ext_vector_type(kPiece / 4)));
  Piece v[kStages][kLoads];

  // stage s of the rows at w (first row, first k of the wave; row_bytes apart)
  __device__ __forceinline__ void load(const uint8_t* w, int row_bytes, int s) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      if constexpr (Q8) {
        int p = 64 * i + lane;
        p = p < 272 ? p : 271;
        const int r = p / 17;
        v[s][i] = *(const GLOBAL_AS Piece*)(w + (size_t)r * row_bytes + kQRow * s +
                                            kPiece * (p - 17 * r));
      } else {
        v[s][i] = load_global(reinterpret_cast<const u32x4*>(
            w + (size_t)(4 * i + (lane >> 4)) * row_bytes + 256 * s + 16 * (lane & 15)));
      }
    }
  }
  __device__ __forceinline__ void stage(uint8_t* slot, int s) const {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      if constexpr (Q8) {
        *reinterpret_cast<Piece*>(slot + kPiece * (64 * i + lane)) = v[s][i];
      } else {
        const int r = 4 * i + (lane >> 4);
        *reinterpret_cast<u32x4*>(slot + 256 * r + 16 * ((lane & 15) ^ r)) = v[s][i];
      }
    }
  }
  // B operand of k block b (32 k) of the staged stage
  static __device__ __forceinline__ f16x8 frag(const uint8_t* slot, int b) {
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, c16 = lane & 15;
    if constexpr (!Q8) {
      return *reinterpret_cast<const f16x8*>(slot + 256 * c16 + 16 * ((4 * b + g) ^ c16));
    } else {
      const uint8_t* wr = slot + kQRow * c16 + 34 * b;
      const _Float16 sc = *reinterpret_cast<const _Float16*>(wr);
      const f16x2 s2 = {sc, sc};
      // the block's int8 k = 8 g .. 8 g + 7 sit at wr + 2 + 8 g: 4-byte
      // aligned for odd b, 2 bytes past a dword boundary for even b
      uint32_t lo, hi;
      if (b % 2 == 0) {
        const uint32_t* p = reinterpret_cast<const uint32_t*>(wr + 8 * g);
        const uint32_t d0 = p[0], d1 = p[1], d2 = p[2];
        lo = __builtin_amdgcn_alignbyte(d1, d0, 2);
        hi = __builtin_amdgcn_alignbyte(d2, d1, 2);
      } else {
        const uint32_t* p = reinterpret_cast<const uint32_t*>(wr + 2 + 8 * g);
        lo = p[0];
        hi = p[1];
      }
      const uint32_t bl = lo ^ 0x80808080u, bh = hi ^ 0x80808080u;
      // exact q in f16, then one rounding of scale * q
      const f16x2 v0 = q8x2_to_f16x2(bl, kSelLo) * s2, v1 = q8x2_to_f16x2(bl, kSelHi) * s2;
      const f16x2 v2 = q8x2_to_f16x2(bh, kSelLo) * s2, v3 = q8x2_to_f16x2(bh, kSelHi) * s2;
      return (f16x8){v0.x, v0.y, v1.x, v1.y, v2.x, v2.y, v3.x, v3.y};
    }
  }
};

template <bool Q8>
constexpr int kRowBytes1024 = Q8 ? 1088 : 2048;  // bytes of 1024 k of a weight row

// Byte offset of row r's 16-byte chunk c in an LDS tile of 1024-column f16
// rows: slot c ^ (r & 15) of each 256 bytes, so a fragment read (16 rows, one
// chunk) touches 16 slots and so does a row write (16 lanes, 16 chunks).
__device__ __forceinline__ int rows_off(int r, int c) { return 2048 * r + 16 * (c ^ (r & 15)); }

// xl rows 0 .. 16 MS - 1 = rms_norm(h[m0 + row], w) (rows past M repeat row
// M - 1).  16 lanes per row, lane p holding chunks p + 16 i, so loads and LDS
// writes are contiguous; the squares are summed in the canonical order (a
// perfect binary tree over the columns in index order: within the chunk, over
// the 16 lanes, over i), so a row's bits are rms_norm's in every other kernel.
// between() runs after the rows have been requested.  out (may be null)
// receives the rows that exist.
template <int MS, int WAVES, class Between>
__device__ __forceinline__ void norm_rows_lds(const uint16_t* h, const uint16_t* w, int m0, int M,
                                              uint8_t* xl, uint16_t* out, Between&& between) {
  const int t = threadIdx.x;
  const int p = t & 15;
  constexpr int kPerPass = 4 * WAVES;  // rows a pass covers
  constexpr int kPasses = (16 * MS + kPerPass - 1) / kPerPass;
  u32x4 hv[kPasses][8], wv[8];
#pragma unroll
  for (int q = 0; q < kPasses; ++q) {
    const int row = kPerPass * q + (t >> 4);
    const int m = m0 + row < M ? m0 + row : M - 1;
    const u32x4* hr = reinterpret_cast<const u32x4*>(h + (size_t)m * kHidden) + p;
#pragma unroll
    for (int i = 0; i < 8; ++i) hv[q][i] = load_global(hr + 16 * i);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) wv[i] = load_global(reinterpret_cast<const u32x4*>(w) + p + 16 * i);
  __builtin_amdgcn_sched_barrier(0);
  between();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < kPasses; ++q) {
    const int row = kPerPass * q + (t >> 4);
    float s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      s[i] = reduce_row16(sq_tree4_mix(hv[q][i][0], hv[q][i][1]) +
                          sq_tree4_mix(hv[q][i][2], hv[q][i][3]));
    const float inv =
        rms_inv(((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7])));
    if (16 * MS % kPerPass == 0 || row < 16 * MS) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        u32x4 x;
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = norm_pair_mix(hv[q][i][j], wv[i][j], inv);
        *reinterpret_cast<u32x4*>(xl + rows_off(row, p + 16 * i)) = x;
        if (out && m0 + row < M)
          reinterpret_cast<u32x4*>(out + (size_t)(m0 + row) * kHidden)[p + 16 * i] = x;
      }
    }
  }
}

// acc[ms] = the products of the LDS rows 16 ms .. + 15 with 16 weight rows
// over 1024 k, one chain of MFMAs in k order.  The first NPRE stages of W have
// been loaded by the caller; the rest are loaded NPRE ahead.
template <bool Q8, int MS, int NPRE>
__device__ __forceinline__ void rows_product(const uint8_t* xl, uint8_t* slot, const uint8_t* w,
                                             WRows<Q8, 1024>& W, f32x4 (&acc)[MS]) {
  using R = WRows<Q8, 1024>;
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, c16 = lane & 15;
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) acc[ms] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int s = 0; s < R::kStages; ++s) {
    W.stage(slot, s);
    if (s + NPRE < R::kStages) W.load(w, kRowBytes1024<Q8>, s + NPRE);
#pragma unroll
    for (int b = 0; b < R::kStageK / 32; ++b) {
      const f16x8 wv = R::frag(slot, b);
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) {
        const f16x8 a = *reinterpret_cast<const f16x8*>(
            xl + rows_off(16 * ms + c16, R::kStageK / 8 * s + 4 * b + g));
        acc[ms] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, wv, acc[ms], 0, 0, 0);
      }
    }
  }
}

struct RowsTile {
  int n_tile, m0;
};
// n tiles in groups of 8, one per XCD; the m tiles of one n tile run on one
// XCD one after another, so its weight rows come from HBM once
__device__ __forceinline__ RowsTile rows_tile(int M, int bm) {
  const int mt = (M + bm - 1) / bm;
  const int slot = blockIdx.x >> 3;
  return RowsTile{(slot / mt) * 8 + (int)(blockIdx.x & 7), (slot % mt) * bm};
}

}  // namespace

// q, k, v of 16 MS tokens for one head (n tile: 0..15 q heads, 16..23 k, 24..31
// v), with everything between the layer's input and its attention:
// xn = rms_norm(h, attn_norm), q/k/v = xn W^T, the heads' norms and RoPE at
// position start + token -> q_roped and the caches.  Wave w owns weight rows
// (head dims) 16 w .. + 15; the head's rows meet in LDS for the norm and RoPE,
// wave w taking tokens w, w + 8, ...
struct RowsQkvArgs {
  const uint16_t* h;
  const uint16_t* norm_w;
  const uint8_t* w[3];  // f16: w[0] the stacked [4096, 1024] matrix; Q8_0: q, k, v layer bases
  uint16_t *xn, *q, *k, *v, *q_roped;
  uint16_t *k_cache, *v_cache;  // the layer's base ([max_seq, 8, 128])
  const uint16_t *qn_w, *kn_w;
  float* rope;  // the RoPE table: read with rope_ready, else written
  int M, start, rope_ready;
};

template <bool Q8, int MS>
__device__ __forceinline__ void rows_qkv(const RowsQkvArgs& A) {
  using W = WRows<Q8, 1024>;
  constexpr int kWaves = 8;
  constexpr int kPre = MS <= 2 ? W::kStages : W::kStages / 2;
  __shared__ __attribute__((aligned(16))) uint8_t xl[16 * MS * 2048];
  __shared__ __attribute__((aligned(16))) uint8_t slots[kWaves * W::kSlot];
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lane = t & 63;
  const int g = lane >> 4, c16 = lane & 15;
  const RowsTile T = rows_tile(A.M, 16 * MS);
  const int kind = T.n_tile < 16 ? 0 : (T.n_tile < 24 ? 1 : 2);  // q, k, v
  const int head = kind == 0 ? T.n_tile : (kind == 1 ? T.n_tile - 16 : T.n_tile - 24);
  const uint8_t* wb = Q8 ? A.w[kind] : A.w[0];
  wb += (size_t)(128 * (Q8 ? head : T.n_tile) + 16 * wave) * kRowBytes1024<Q8>;
  W wr;
  norm_rows_lds<MS, kWaves>(A.h, A.norm_w, T.m0, A.M, xl, T.n_tile == 0 ? A.xn : nullptr, [&] {
#pragma unroll
    for (int i = 0; i < kPre; ++i) wr.load(wb, kRowBytes1024<Q8>, i);
  });
  // the angles of this wave's 2 MS tokens (wave, wave + 8, ...), while the
  // weights are in flight; a half wave computes one token's 64 frequencies
  constexpr int R = 2 * MS;
  float cs[R][2], sn[R][2];
  if (kind != 2) {
    if (A.rope_ready) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int m = T.m0 + wave + 8 * i < A.M ? T.m0 + wave + 8 * i : A.M - 1;
        rope_lane(A.rope, m, cs[i], sn[i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < R; i += 2) {
        const int tok = T.m0 + wave + 8 * (i + (lane >> 5));
#pragma unroll
        for (int dd = 0; dd < 2; ++dd) {
          float c, s;
          rope_angle(A.start + tok, (2 * lane + dd) & 63, c, s);
          const float co = xor32(c), so = xor32(s);
          cs[i][dd] = lane < 32 ? c : co;
          sn[i][dd] = lane < 32 ? s : so;
          cs[i + 1][dd] = lane < 32 ? co : c;
          sn[i + 1][dd] = lane < 32 ? so : s;
          if (T.n_tile == 0 && tok < A.M) {
            A.rope[(size_t)tok * 128 + ((2 * lane + dd) & 63)] = c;
            A.rope[(size_t)tok * 128 + 64 + ((2 * lane + dd) & 63)] = s;
          }
        }
      }
    }
  }
  const f16x2 nw = as_f16x2(load_global(
      reinterpret_cast<const uint32_t*>(kind == 0 ? A.qn_w : A.kn_w) + lane));
  __syncthreads();
  f32x4 acc[MS];
  rows_product<Q8, MS, kPre>(xl, slots + W::kSlot * wave, wb, wr, acc);
  __syncthreads();
  // the head's rows over the token tile: [16 MS][128] f16, 272 bytes a row
  constexpr int kRow = 272;
#pragma unroll
  for (int ms = 0; ms < MS; ++ms)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<uint16_t*>(xl + (16 * ms + 4 * g + i) * kRow + 2 * (16 * wave + c16)) =
          f32_to_f16_bits(acc[ms][i]);
  __syncthreads();
  uint16_t* raw = kind == 0 ? A.q : (kind == 1 ? A.k : A.v);
  const int ld = kind == 0 ? 2048 : 1024;
  uint32_t xw[R], out[R];
#pragma unroll
  for (int i = 0; i < R; ++i)
    xw[i] = *reinterpret_cast<const uint32_t*>(xl + (wave + 8 * i) * kRow + 4 * lane);
  if (kind != 2) {
#pragma unroll
    for (int i = 0; i < R; ++i) out[i] = head_norm_rope(xw[i], nw, cs[i], sn[i]);
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int m = T.m0 + wave + 8 * i;
    if (m < A.M) {
      reinterpret_cast<uint32_t*>(raw + (size_t)m * ld + head * kHeadDim)[lane] = xw[i];
      const size_t slot = ((size_t)(A.start + m) * kKvHeads + head) * kHeadDim;
      if (kind == 0)
        reinterpret_cast<uint32_t*>(A.q_roped + (size_t)m * 2048 + head * kHeadDim)[lane] = out[i];
      else if (kind == 1)
        reinterpret_cast<uint32_t*>(A.k_cache + slot)[lane] = out[i];
      else
        reinterpret_cast<uint32_t*>(A.v_cache + slot)[lane] = xw[i];
    }
  }
}

// rms_norm and the product behind it for 16 MS tokens: q, k and v (16 NS of the
// 4096 output columns per workgroup) or gate/up with SwiGLU (8 NS outputs, 16
// gate and the matching 16 up rows in turn).  Eight waves split K = 1024: wave
// w holds k 128 w .. + 127 of the token rows and of its weight rows, everything
// requested at once; the row's square sums meet in LDS (the canonical order:
// 8 columns, 16 lanes, 8 waves), then the eight ranges' products are added in
// order.
struct RowsNormArgs {
  const uint16_t* h;
  const uint16_t* norm_w;
  const uint8_t* w[3];  // f16: w[0]; Q8_0: q, k, v layer bases, or w[0] the gate/up stack
  uint16_t* x;          // the normalised rows
  uint16_t* y[3];       // q, k, v; or y[0] the SwiGLU output
  float* rope;          // the RoPE table of positions start + token, written if not null
  int M, start;
};

template <bool GU, bool Q8, int MS, int NS>
__device__ __forceinline__ void rows_norm(const RowsNormArgs& A) {
  static_assert(!GU || NS % 2 == 0, "gate/up pairs");
  using W = WRows<Q8, 128>;
  constexpr int kWaves = 8;
  constexpr int kSlot = W::kSlot > 4096 ? W::kSlot : 4096;
  constexpr int kRed = kWaves * MS * NS * 1024;
  constexpr int kLds = 2 * kWaves * kSlot > kRed ? 2 * kWaves * kSlot : kRed;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kLds];
  __shared__ __attribute__((aligned(16))) float ss[16 * MS][kWaves];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, c16 = lane & 15;
  const RowsTile T = rows_tile(A.M, 16 * MS);
  constexpr int kRowBytes = kRowBytes1024<Q8>;

  u32x4 hv[MS][4];  // row 16 ms + 4 i + g, columns 128 wave + 8 c16 .. + 7
#pragma unroll
  for (int ms = 0; ms < MS; ++ms)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = T.m0 + 16 * ms + 4 * i + g;
      const int m = row < A.M ? row : A.M - 1;
      hv[ms][i] = load_global(
          reinterpret_cast<const u32x4*>(A.h + (size_t)m * kHidden + 128 * wave) + c16);
    }
  const u32x4 nw = load_global(reinterpret_cast<const u32x4*>(A.norm_w + 128 * wave) + c16);
  // first output column (q/k/v: within q, k or v; gate/up: SwiGLU outputs)
  // and the weight rows of its 16-row groups
  const int first = 16 * NS * T.n_tile;
  const int seg = GU ? 0 : (first < 2048 ? 0 : (first < 3072 ? 1 : 2));
  const int col0 = GU ? first / 2 : (seg == 0 ? first : first - 1024 - 1024 * seg);
  W wr[NS];
#pragma unroll
  for (int ns = 0; ns < NS; ++ns) {
    int row;
    if constexpr (GU && Q8) row = kFfn * (ns & 1) + col0 + 16 * (ns >> 1);
    else row = (Q8 ? col0 : first) + 16 * ns;
    wr[ns].load((Q8 ? A.w[seg] : A.w[0]) + (size_t)row * kRowBytes + kRowBytes / 8 * wave,
                kRowBytes, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
  // the RoPE table, spread over the workgroups of the first token tile
  if (!GU && A.rope != nullptr && T.m0 == 0) {
    for (int tok = T.n_tile + 256 / NS * wave; tok < A.M; tok += 256 / NS * kWaves) {
      float c, s;
      rope_angle(A.start + tok, lane, c, s);
      A.rope[(size_t)tok * 128 + lane] = c;
      A.rope[(size_t)tok * 128 + 64 + lane] = s;
    }
  }
#pragma unroll
  for (int ms = 0; ms < MS; ++ms)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x4 v = hv[ms][i];
      const float q = reduce_row16(sq_tree4_mix(v[0], v[1]) + sq_tree4_mix(v[2], v[3]));
      if (c16 == 0) ss[16 * ms + 4 * i + g][wave] = q;
    }
  __syncthreads();
  // 1 / rms of row `lane` of the tile in this lane, handed to the lanes that
  // hold the row's columns by ds_bpermute below
  float inv_row;
  {
    const float* sr = ss[lane & (16 * MS - 1)];
    const f32x4 s0 = *reinterpret_cast<const f32x4*>(sr);
    const f32x4 s1 = *reinterpret_cast<const f32x4*>(sr + 4);
    inv_row = rms_inv(((s0[0] + s0[1]) + (s0[2] + s0[3])) + ((s1[0] + s1[1]) + (s1[2] + s1[3])));
  }
  // the wave's two LDS slots in turn: LDS operations of one wave complete in
  // order, so a slot may be written again once its reads have been issued
  uint8_t* slot = lds + 2 * kSlot * wave;
  f16x8 wf[NS][4];
#pragma unroll
  for (int ns = 0; ns < NS; ++ns) {
    wr[ns].stage(slot + kSlot * (ns & 1), 0);
#pragma unroll
    for (int b = 0; b < 4; ++b) wf[ns][b] = W::frag(slot + kSlot * (ns & 1), b);
  }
  f32x4 acc[MS][NS];
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) {
    uint8_t* xs = slot + kSlot * ((NS + ms) & 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * i + g;
      const float inv = __uint_as_float(
          __builtin_amdgcn_ds_bpermute(4 * (16 * ms + row), __float_as_uint(inv_row)));
      u32x4 x;
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = norm_pair_mix(hv[ms][i][j], nw[j], inv);
      *reinterpret_cast<u32x4*>(xs + 256 * row + 16 * (c16 ^ row)) = x;
      const int m = T.m0 + 16 * ms + row;
      if (T.n_tile == 0 && m < A.M)
        reinterpret_cast<u32x4*>(A.x + (size_t)m * kHidden + 128 * wave)[c16] = x;
    }
#pragma unroll
    for (int ns = 0; ns < NS; ++ns) acc[ms][ns] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const f16x8 a = *reinterpret_cast<const f16x8*>(xs + 256 * c16 + 16 * ((4 * b + g) ^ c16));
#pragma unroll
      for (int ns = 0; ns < NS; ++ns)
        acc[ms][ns] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, wf[ns][b], acc[ms][ns], 0, 0, 0);
    }
  }
  __syncthreads();
  f32x4* red = reinterpret_cast<f32x4*>(lds);
#pragma unroll
  for (int ms = 0; ms < MS; ++ms)
#pragma unroll
    for (int ns = 0; ns < NS; ++ns) red[((wave * MS + ms) * NS + ns) * 64 + lane] = acc[ms][ns];
  __syncthreads();
  // wave w finishes output tiles w, w + 8, ... (16 tokens x 16 outputs each)
  constexpr int NO = GU ? NS / 2 : NS;  // output tiles across
  constexpr int NI = GU ? 2 : 1;        // 16-row weight groups per output tile
#pragma unroll
  for (int u0 = 0; u0 < MS * NO; u0 += kWaves) {
    const int u = u0 + wave;
    if (MS * NO % kWaves == 0 || u < MS * NO) {
      const int ms = u / NO, no = u - ms * NO;
      f32x4 a[NI];
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int at = (ms * NS + NI * no + j) * 64 + lane;
        a[j] = red[at];
#pragma unroll
        for (int s = 1; s < kWaves; ++s) a[j] += red[s * MS * NS * 64 + at];
      }
      const int ld = GU ? kFfn : (seg == 0 ? 2048 : 1024);
      uint16_t* y = A.y[seg] + col0 + 16 * no + c16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = T.m0 + 16 * ms + 4 * g + i;
        if (m < A.M)
          y[(size_t)m * ld] = GU ? swiglu_f16(a[0][i], a[NI - 1][i]) : f32_to_f16_bits(a[0][i]);
      }
    }
  }
}

// y = r + x W^T for 16 MS tokens and 16 of the 1024 outputs (attn_o, ffn_down):
// wave w multiplies k 256 w .. + 255, x and weight fragments both straight
// from memory (no two waves share either), and the K / 256 ranges' sums are
// added through LDS in order.
struct RowsResArgs {
  const uint16_t* x;  // [M, K]
  const uint8_t* w;   // [1024, K]
  const uint16_t* r;
  uint16_t* y;
  int M;
};

template <bool Q8, int MS, int WAVES>
__device__ __forceinline__ void rows_res(const RowsResArgs& A) {
  constexpr int K = 256 * WAVES;
  using W = WRows<Q8, 256>;
  constexpr int kXSlot = 16 * MS * 256;  // 128 k of the token rows
  constexpr int kLds = WAVES * (W::kSlot + kXSlot);
  __shared__ __attribute__((aligned(16))) uint8_t lds[kLds];
  static_assert(kLds >= WAVES * MS * 1024, "partial sums");
  f32x4* red = reinterpret_cast<f32x4*>(lds);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, c16 = lane & 15;
  const RowsTile T = rows_tile(A.M, 16 * MS);
  const int n0 = 16 * T.n_tile;
  constexpr int kRowBytes = kRowBytes1024<Q8> / 4 * WAVES;
  const uint8_t* wb = A.w + (size_t)n0 * kRowBytes + kRowBytes1024<Q8> / 4 * wave;
  uint8_t* wslot = lds + (W::kSlot + kXSlot) * wave;
  uint8_t* xslot = wslot + W::kSlot;
  W wr;
#pragma unroll
  for (int s = 0; s < W::kStages; ++s) wr.load(wb, kRowBytes, s);
  u32x4 xv[2][4 * MS];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4 * MS; ++i) {
      const int row = 4 * i + (lane >> 4);
      const int m = T.m0 + row < A.M ? T.m0 + row : A.M - 1;
      xv[h][i] = load_global(
          reinterpret_cast<const u32x4*>(A.x + (size_t)m * K + 256 * wave + 128 * h) + c16);
    }
  // the residuals of the outputs this wave will finish (token tile `wave`)
  uint16_t rv[4];
  if (wave < MS) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = T.m0 + 16 * wave + 4 * g + i < A.M ? T.m0 + 16 * wave + 4 * g + i : A.M - 1;
      rv[i] = load_global_u16(A.r + (size_t)m * kHidden + n0 + c16);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  f32x4 acc[MS];
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) acc[ms] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (h < W::kStages) wr.stage(wslot, h);
#pragma unroll
    for (int i = 0; i < 4 * MS; ++i) {
      const int row = 4 * i + (lane >> 4);
      *reinterpret_cast<u32x4*>(xslot + 256 * row + 16 * (c16 ^ (row & 15))) = xv[h][i];
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const f16x8 wv = W::frag(wslot, Q8 ? 4 * h + b : b);
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) {
        const f16x8 a = *reinterpret_cast<const f16x8*>(xslot + 256 * (16 * ms + c16) +
                                                        16 * ((4 * b + g) ^ c16));
        acc[ms] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, wv, acc[ms], 0, 0, 0);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) red[(wave * MS + ms) * 64 + lane] = acc[ms];
  __syncthreads();
  if (wave < MS) {
    f32x4 a = red[wave * 64 + lane];
#pragma unroll
    for (int s = 1; s < WAVES; ++s) a += red[(s * MS + wave) * 64 + lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = T.m0 + 16 * wave + 4 * g + i;
      if (m < A.M) A.y[(size_t)m * kHidden + n0 + c16] = residual_f16(as_half(rv[i]), a[i]);
    }
  }
}

// Instances by 16-token tiles (and, for the products behind a norm, 16-row
// weight groups) per workgroup; the host's rows_* launchers say which serves
// how many tokens.
#define PF_ROWS(name, threads, Args, ...) \
  extern "C" __global__ __launch_bounds__(threads) void name(Args A) { __VA_ARGS__(A); }
PF_ROWS(pf_rows_qkv_rope, 512, RowsQkvArgs, rows_qkv<false, 1>)
PF_ROWS(pf_rows_qkv_rope_q8, 512, RowsQkvArgs, rows_qkv<true, 1>)
#define PF_ROWS_QKV(MS, NS)                                                                  \
  PF_ROWS(pf_rows_qkv_##MS##NS, 512, RowsNormArgs, rows_norm<false, false, MS, NS>)          \
  PF_ROWS(pf_rows_qkv_q8_##MS##NS, 512, RowsNormArgs, rows_norm<false, true, MS, NS>)
PF_ROWS_QKV(1, 1)
PF_ROWS_QKV(1, 2)
#define PF_ROWS_GU(MS, NS)                                                                   \
  PF_ROWS(pf_rows_gu_##MS##NS, 512, RowsNormArgs, rows_norm<true, false, MS, NS>)            \
  PF_ROWS(pf_rows_gu_q8_##MS##NS, 512, RowsNormArgs, rows_norm<true, true, MS, NS>)
PF_ROWS_GU(1, 2)
PF_ROWS_GU(2, 2)
PF_ROWS_GU(2, 4)
PF_ROWS_GU(2, 6)
#define PF_ROWS_RES(MS)                                                                      \
  PF_ROWS(pf_rows_o_##MS, 512, RowsResArgs, rows_res<false, MS, 8>)                          \
  PF_ROWS(pf_rows_o_q8_##MS, 512, RowsResArgs, rows_res<true, MS, 8>)                        \
  PF_ROWS(pf_rows_dn_##MS, 768, RowsResArgs, rows_res<false, MS, 12>)                        \
  PF_ROWS(pf_rows_dn_q8_##MS, 768, RowsResArgs, rows_res<true, MS, 12>)
PF_ROWS_RES(1)
PF_ROWS_RES(2)
#undef PF_ROWS_QKV
#undef PF_ROWS_GU
#undef PF_ROWS_RES
#undef PF_ROWS

#endif
