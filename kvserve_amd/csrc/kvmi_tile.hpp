// Wave-tile kernels: paged compress / decompress of the geometries and options that the
// kernels of kvmi_mfma.hip do not take -- head sizes that are not 64 or 128 (80, 96, 112,
// 160, 192, 224, and 256 where the paired view does not apply), head counts that do not
// divide 8, the other quantization axes, and the pipeline without the transform.
//
// Tile.  A wave owns whole tokens: a tile is T = min(32 / H, S) tokens x H heads, row
// r = token * H + head, so a lane keeps its head for the whole kernel and a tile touches
// at most two paged blocks; with H = 6 it fills 30 of the 32 MFMA columns.  The rows are
// loaded in 16-byte pieces, lane-linear (1 KiB an instruction), and turned into MFMA
// operands through the wave's own LDS buffer.
//
// Transform.  A head of D channels is the reference's descending power-of-two chunks
// (hadamard_func.py:50-103), so its matrix is block diagonal.  With input e = 16 s + 8 hl
// + j and output f = 32 c + 16 hl + i (see hadamard_tile_d) every 32 x 16 tile inside a
// chunk is +-1 times one of two base tiles, and tiles between chunks are skipped: D = 96
// takes 10 products for its 3 output tiles.  A last chunk of 16 channels fills the lower
// lane half of its tile; the upper half then holds a copy that is never stored.
//
// Waves do not wait for each other: a wave packs NT tiles of one part into its own LDS
// image, one run of NT * T tokens per head (permuted order), and writes the runs in
// 16-byte pieces; decode reads them the same way.  The only workgroup barriers are those
// behind the table set-up.  4 bits has kernels of its own; the other widths share one per head
// size, with the width a kernel argument (a uniform branch per 16 symbols).
#pragma once

#include <type_traits>

#include "kvmi_mfma_tiles.hpp"

namespace kvmi {

// Launch shape, computed on the host (kvmi_tile_stats.hip: tile_plan).
struct TileArgs {
  int T;           // tokens per tile
  int ST;          // tokens per super-tile: NT tiles of one wave
  int run;         // tokens per workgroup
  int pitch;       // bytes of one run (head) in a wave's packed image
  int runs;        // runs in an image: H (permuted), 1 (native)
  uint32_t magic;  // floor(2^32 / S) + 1, or 0 for S = 1
  int tabs;        // bit p: part p takes its constants from a table (channel / tensor axis)
  int off_tab;     // byte offsets of the dynamic LDS: constant tables, wave buffers
  int off_wave;
  int wave_bytes;  // tile buffer + packed image of one wave
  int parts;       // parts a workgroup takes: 2, or 1 (blockIdx.z) in small launches
};

constexpr int kTileMaxH = 32;
constexpr int kTileWaves = 4;
constexpr int kTileThreads = 64 * kTileWaves;

// Waves per SIMD the registers of the encode and decode kernels are limited to.
constexpr int tile_occ(int D) { return D <= 128 ? 3 : 2; }
TileArgs tile_plan(const Geo& g, int32_t max_blocks, int32_t num_jobs, int occ);
int tile_cus();

namespace {

// ---------------------------------------------------------------- head size
constexpr int tile_chunk_start(int D, int ch) {
  int st = 0;
  for (int b = 8; b >= 4; --b) {
    const int c = 1 << b;
    if (!(D & c)) continue;
    if (ch < st + c) return st;
    st += c;
  }
  return st;
}
constexpr int tile_chunk_size(int D, int ch) {
  int st = 0;
  for (int b = 8; b >= 4; --b) {
    const int c = 1 << b;
    if (!(D & c)) continue;
    if (ch < st + c) return c;
    st += c;
  }
  return 16;
}
// fp32 value of 1 / sqrt(c) for c = 16 .. 256, rounded once from double
constexpr float tile_chunk_scale(int c) {
  double s = 1.0;
  int x = c;
  while (x >= 4) {
    s *= 0.5;
    x /= 4;
  }
  return (float)(x == 2 ? s * 0.70710678118654752440 : s);
}

template <int D>
struct TileGeo {
  static_assert(D % 16 == 0 && D >= 16 && D <= 256, "whole 16-channel steps");
  static constexpr int KS = D / 16;         // 16-channel input steps of a row
  static constexpr int NC = (D + 31) / 32;  // 32-channel output tiles
  static constexpr int PR = D / 8;          // 16-byte pieces of a row
  // The wave's buffer holds 64 channels of the 32 rows at a time where the row is a multiple
  // of 128 bytes (whole cache lines either way; at D = 128 the buffer is 4.6 KB instead of
  // 8.7 and 12 waves fit a CU instead of 8), else whole rows.
  static constexpr bool kHalves = D % 64 == 0;
  static constexpr int NG = kHalves ? D / 64 : 1;  // groups a row is staged in
  static constexpr int PG = PR / NG;               // pieces of a row in a group
  static constexpr int KG = KS / NG;               // load / store instructions of a group
  static constexpr int PP = PG + 1;                // LDS pitch of a row, in pieces
  static constexpr int kBuf = kTok * PP;           // uint4 of a wave's tile buffer
  static constexpr bool kTail = D % 32 == 16;
};

// Is the lane half hl of output tile cp part of the row?
template <int D, int CP>
__device__ __forceinline__ bool tile_half_ok(int hl) {
  return !(TileGeo<D>::kTail && CP == TileGeo<D>::NC - 1) || hl == 0;
}

// f(integral_constant<0>), ..., f(integral_constant<N - 1>): loops over output tiles whose
// index has to be a constant (the products of a tile depend on its chunk).
template <int N, int I = 0, class F>
__device__ __forceinline__ void tile_each(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    tile_each<N, I + 1>(f);
  }
}

// Output tile CP (unscaled fp32) of the row operands x[s]: mul(base tile, operand, sum) of
// every input step of its chunk.  The chunk's 32-channel inputs are visited in the order
// own ^ k, so the sums of different output tiles share no prefix (see transform_T).
template <int D, int CP, class Mul>
__device__ __forceinline__ f32x16 tile_transform(const uint4 (&x)[2 * TileGeo<D>::NC], const uint4 (&hp)[2], const uint4 (&hn)[2],
                                                 Mul mul) {
  constexpr int c0 = tile_chunk_start(D, 32 * CP), cs = tile_chunk_size(D, 32 * CP), own = CP - c0 / 32;
  f32x16 acc = {};
  if constexpr (cs == 16) {
    acc = mul(hp[0], x[c0 / 16], acc);
  } else {
#pragma unroll
    for (int k = 0; k < cs / 32; ++k) {
      const int t = own ^ k;
      const bool neg = __builtin_popcount(own & t) & 1;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) acc = mul(neg ? hn[kt] : hp[kt], x[c0 / 16 + 2 * t + kt], acc);
    }
  }
  return acc;
}
template <int D, int CP>
constexpr float kTileScale = tile_chunk_scale(tile_chunk_size(D, 32 * CP));

// ---------------------------------------------------------------- addresses
__device__ __forceinline__ int tile_block_of(int tok, const TileArgs& a) {
  return a.magic ? (int)__umulhi((uint32_t)tok, a.magic) : tok;
}

// The rows of a tile in the pool: `n` tokens from token `ta`, in one block or two.  Row i
// starts at base0 + i rows in the first block and at base1 + i rows in the second.
struct TileRows {
  uint64_t base0, base1;
  int n0, nr;  // rows in the first block, rows in all
};
template <int D>
__device__ __forceinline__ TileRows tile_rows(const kvmi_layer_job& job, const Geo& g, const TileArgs& a, int part,
                                              int ta, int n) {
  const int S = g.S, HD = g.H * D;
  const int b0 = tile_block_of(ta, a), off = ta - b0 * S;
  const uint64_t pool = (uint64_t)(reinterpret_cast<uint16_t*>(job.pool) + (part ? job.pool_part_stride : 0));
  TileRows t;
  t.nr = n * g.H;
  t.n0 = min(n, S - off) * g.H;
  t.base0 = pool + 2u * (((int64_t)cld(job.block_ids + b0) * S + off) * HD);
  t.base1 = pool + 2u * ((int64_t)cld(job.block_ids + min(b0 + 1, job.num_blocks - 1)) * S * HD - (int64_t)t.n0 * D);
  return t;
}
// Instruction v of the tile moves the lane's 16-byte piece of (row, col): lane-linear over
// the rows of a group, groups one after the other.
template <int D>
__device__ __forceinline__ int tile_row_of(int v, int l) {
  return (64 * (v % TileGeo<D>::KG) + l) / TileGeo<D>::PG;
}
template <int D>
__device__ __forceinline__ int tile_col_of(int v, int l) {
  return (64 * (v % TileGeo<D>::KG) + l) % TileGeo<D>::PG + v / TileGeo<D>::KG * TileGeo<D>::PG;
}
// Its index in the pool's pieces, from the tile's first row, and in the wave's buffer.
template <int D>
__device__ __forceinline__ uint32_t tile_index(int v, int l) {
  if constexpr (!TileGeo<D>::kHalves) return (uint32_t)(64 * v + l);
  return (uint32_t)(tile_row_of<D>(v, l) * TileGeo<D>::PR + tile_col_of<D>(v, l));
}
template <int D>
__device__ __forceinline__ int tile_slot_of(int v, int l) {
  using TG = TileGeo<D>;
  if constexpr (!TG::kHalves) return 64 * v + l + (64 * v + l) / TG::PG;
  return tile_row_of<D>(v, l) * TG::PP + (l % TG::PG);
}
// All pieces of the tile (past its end its last row, or last piece, again: not used).  A
// tile of 32 rows in one block takes scalar-base addresses.
template <int D>
__device__ __forceinline__ void tile_load(const TileRows& t, int l, uint4 (&x)[D / 16]) {
  using TG = TileGeo<D>;
  const uint4* b = reinterpret_cast<const uint4*>(t.base0);
  if (t.n0 == kTok) {
#pragma unroll
    for (int v = 0; v < TG::KS; ++v) x[v] = gld(b + tile_index<D>(v, l));
    return;
  }
  if constexpr (TG::kHalves) {
    const int last = t.nr - 1;
#pragma unroll
    for (int v = 0; v < TG::KS; ++v) {
      const int row = min(tile_row_of<D>(v, l), last);
      const uint64_t base = row < t.n0 ? t.base0 : t.base1;
      x[v] = gld(reinterpret_cast<const uint4*>(base) + (uint32_t)(row * TG::PR + tile_col_of<D>(v, l)));
    }
  } else {
    const int last = t.nr * TG::PR - 1, p0 = t.n0 * TG::PR;
#pragma unroll
    for (int v = 0; v < TG::KS; ++v) {
      const int p = min(64 * v + l, last);
      const uint64_t base = p < p0 ? t.base0 : t.base1;
      x[v] = gld(reinterpret_cast<const uint4*>(base) + (uint32_t)p);
    }
  }
}
// Store group gi of the tile's rows from the wave's buffer.
template <int D>
__device__ __forceinline__ void tile_store(const TileRows& t, int gi, int l, const uint4* tb) {
  using TG = TileGeo<D>;
  uint4* b = reinterpret_cast<uint4*>(t.base0);
  if (t.n0 == kTok) {
#pragma unroll
    for (int v = gi * TG::KG; v < (gi + 1) * TG::KG; ++v) gst_stream(b + tile_index<D>(v, l), tb[tile_slot_of<D>(v, l)]);
    return;
  }
#pragma unroll
  for (int v = gi * TG::KG; v < (gi + 1) * TG::KG; ++v) {
    const int p = TG::kHalves ? tile_row_of<D>(v, l) : 64 * v + l;
    const int n = TG::kHalves ? t.nr : t.nr * TG::PR, n0 = TG::kHalves ? t.n0 : t.n0 * TG::PR;
    if (p < n) {
      const uint64_t base = p < n0 ? t.base0 : t.base1;
      gst_stream(reinterpret_cast<uint4*>(base) + tile_index<D>(v, l), tb[tile_slot_of<D>(v, l)]);
    }
  }
}

// Byte offset of run j's token `tok` in the job's packed stream behind its header.
__device__ __forceinline__ uint8_t* tile_stream(const kvmi_layer_job& job, const Geo& g, int part, int j, int tok,
                                                int ntok, int RB) {
  uint8_t* s = job.stream + ((g.flags & KVMI_F_NO_HEADER) ? 0 : KVMI_HEADER_BYTES) + job.symbol_offset * g.bits / 8;
  const int64_t row = (g.flags & KVMI_F_NATIVE_LAYOUT) ? ((int64_t)part * ntok + tok) * g.H
                                                       : ((int64_t)part * g.H + j) * ntok + tok;
  return s + row * RB;
}

// Packed symbols are written and read at several widths and at addresses that are a
// multiple of 2 only (rows of odd widths), or of nothing (8 symbols of one).
typedef uint16_t __attribute__((may_alias)) u16any;
struct __attribute__((packed, aligned(2), may_alias)) Bytes16 {
  uint32_t x, y, z, w;
};
struct __attribute__((packed, aligned(1), may_alias)) Word1 {
  uint32_t v;
};
struct __attribute__((packed, aligned(1), may_alias)) Word2 {
  uint32_t a, b;
};
__device__ __forceinline__ uint4 ld16u(const uint8_t* p) {
  const KVMI_GLOBAL Bytes16* q = (const KVMI_GLOBAL Bytes16*)p;
  return make_uint4(q->x, q->y, q->z, q->w);
}
__device__ __forceinline__ void st16u(uint8_t* p, uint4 v) {
  KVMI_GLOBAL Bytes16* q = (KVMI_GLOBAL Bytes16*)p;
  q->x = v.x;
  q->y = v.y;
  q->z = v.z;
  q->w = v.w;
}

// The packed bytes of a super-tile: `runs` runs of `rl` bytes, run j at j * stride behind
// the first in the stream and at j * pitch in the image, moved in 16-byte slots (a run's
// last slot ends with the run and may overlap the one before it).
struct TileSlots {
  int rl, ns, count;
  float inv;
};
__device__ __forceinline__ TileSlots tile_slots(int rl, int runs) {
  TileSlots s;
  s.rl = rl;
  s.ns = (rl + 15) >> 4;
  s.count = runs * s.ns;
  s.inv = 1.0f / (float)s.ns;
  return s;
}
__device__ __forceinline__ void tile_slot(const TileSlots& s, int q, int& j, int& off) {
  j = (int)(((float)q + 0.5f) * s.inv);
  off = min(16 * (q - (int)__umul24(j, s.ns)), s.rl - 16);
}

// ---------------------------------------------------------------- per-workgroup tables
struct TileTables {
  uint8_t prof[2][3][kTileMaxH];  // the job's profile bytes
  uint8_t pos[2][kTileMaxH];      // output position of each source head
  // token-axis statistics by source head: the head each reduction step reads (bytes 0 - 4),
  // the group (5) and whether the head is the group's first output position (6)
  uint2 group[2][kTileMaxH];
};

__device__ __forceinline__ void tile_stage_profile(TileTables& T, const uint8_t* profile, int H) {
  for (int i = threadIdx.x; i < 6 * H; i += kTileThreads) T.prof[i / (3 * H)][(i / H) % 3][i % H] = gld(profile + i);
}
// Output positions (behind a barrier after the profile).
__device__ __forceinline__ void tile_positions(TileTables& T, int H) {
  for (int i = threadIdx.x; i < 2 * H; i += kTileThreads) {
    const int part = i / H, k = i % H;
    T.pos[part][T.prof[part][0][k]] = (uint8_t)k;
  }
}
// Groups of the parts on the token axis (those without a bit in `tabs`), for encode alone.  The
// reduction over the n heads of a group visits members (m + 1) % n, (m + 2) % n, (m + 4) % n,
// ... of head m's own token: min and max may count a member twice.
__device__ __forceinline__ void tile_groups(TileTables& T, int H, int tabs) {
  for (int i = threadIdx.x; i < 2 * H; i += kTileThreads) {
    const int part = i / H, k = i % H, h = T.prof[part][0][k], grp = T.prof[part][2][k];
    if ((tabs >> part) & 1) continue;
    int m = 0, n = 0;
    for (int c = 0; c < H; ++c) {
      if (T.prof[part][2][c] != grp) continue;
      if (c == k) m = n;
      ++n;
    }
    uint32_t lo = 0, hi = (uint32_t)grp << 8 | (m == 0 ? 1u << 16 : 0u);
    int at = 0;
    for (int c = 0; c < H; ++c) {
      if (T.prof[part][2][c] != grp) continue;
      const uint32_t src = T.prof[part][0][c];
      const int d = at - m + (at < m ? n : 0);  // steps from m to this member
      // a step of 2^b reaches (m + 2^b) % n; past one lap the head itself is as good
      if (d == 1 % n) lo |= src;
      if (d == 2 % n) lo |= src << 8;
      if (d == 4 % n) lo |= src << 16;
      if (d == 8 % n) lo |= src << 24;
      if (d == 16 % n) hi |= src;
      ++at;
    }
    T.group[part][h] = make_uint2(lo, hi);
  }
}
// The tables below are read from memory in one trip each: a loop of single loads that wait for
// each other was half of a short call (4 layers x 768 tokens x 30 heads of 64 at 6 bits, both
// parts by channel: encode 37 -> 20 us, decode 33 -> 21; a request of 16 x 4080 x 6 x 96 decodes in
// 44 us instead of 49).
//
// Sign masks: row of D / 2 words (+ 4 of padding) per head, word p flips elements 2p, 2p + 1.
template <int D>
__device__ __forceinline__ void tile_signs(uint32_t* smask, const uint32_t* signs, int H) {
  constexpr int W = (D + 31) / 32;  // words of signs a head
  for (int i = threadIdx.x; i < H * W; i += kTileThreads) {
    const int h = i / W, w = i % W;
    const uint32_t s = gld(signs + i);
    uint4* row = reinterpret_cast<uint4*>(smask + h * (D / 2 + 4) + 16 * w);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (D % 32 == 16 && w == W - 1 && q >= 2) break;
      uint32_t m[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const uint32_t t = s >> (8 * q + 2 * p);
        m[p] = ((t & 1u) << 15) | ((t & 2u) << 30);
      }
      row[q] = make_uint4(m[0], m[1], m[2], m[3]);
    }
  }
}
// Constants of a channel- or tensor-axis part by source head and channel: (min, -1 / scale)
// for encode, (min, scale) for decode.  8 channels a thread; the tables of a part are at
// multiples of 2 bytes.
template <int D, bool DIV>
__device__ __forceinline__ void tile_consts(float2* kc, const TileTables& T, const Geo& g, const uint16_t* meta,
                                            int part) {
  const int HD = g.H * D;
  const bool channel = part_axis(g.flags, part) == kAxChannel;
  for (int i = threadIdx.x; i < HD / 8; i += kTileThreads) {
    const int j = i / (D / 8), e = i % (D / 8) * 8;
    uint4 mn, sc;
    if (channel) {
      mn = ld16u(reinterpret_cast<const uint8_t*>(meta + 8 * i));
      sc = ld16u(reinterpret_cast<const uint8_t*>(meta + HD + 8 * i));
    } else {
      const int grp = T.prof[part][2][j];
      const uint32_t a = gld(meta + grp) * 0x10001u, b = gld(meta + g.G + grp) * 0x10001u;
      mn = make_uint4(a, a, a, a);
      sc = make_uint4(b, b, b, b);
    }
    const uint32_t m[4] = {mn.x, mn.y, mn.z, mn.w}, s[4] = {sc.x, sc.y, sc.z, sc.w};
    float4* to = reinterpret_cast<float4*>(kc + T.prof[part][0][j] * (D + 4) + e);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const float s0 = bf_lo(s[p]), s1 = bf_hi(s[p]);
      to[p] = make_float4(bf_lo(m[p]), DIV ? -1.0f / s0 : s0, bf_hi(m[p]), DIV ? -1.0f / s1 : s1);
    }
  }
}

// Min / max over the heads of the lane's group (TileTables::group) and both lane halves;
// `lane0` is the lane of head 0 of the lane's token.
__device__ __forceinline__ void tile_group_minmax(uint2 grp, int lane0, int H, float& a, float& b) {
  a = halves_min(a);
  b = halves_max(b);
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    if ((1 << k) >= H) break;
    const int src = 4 * (lane0 + (int)(((k < 4 ? grp.x : grp.y) >> (8 * (k & 3))) & 0xffu));
    a = fminf(a, __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(a))));
    b = fmaxf(b, __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(b))));
  }
}

}  // namespace
}  // namespace kvmi
