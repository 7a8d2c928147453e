// Statistics pass of the wave-tile kernels (kvmi_tile.hpp) for the parts on the channel or
// tensor axis, and the launch shape of all three passes.
#include <algorithm>

#include "kvmi_tile.hpp"

namespace kvmi {
namespace {

constexpr int kStatTok = 32;  // tokens of a statistics tile

// A tile is 32 consecutive tokens of one head (rows 2 H D bytes apart; past the run its last
// token again, which min and max ignore), transformed in orientation N: a lane holds 16
// rows of one channel, so a head's running minimum and maximum are one pair per output tile.
// The (head, tile) pairs of a run are split evenly over the waves of its workgroups (several in
// short calls, blockIdx.z), head by head; where a wave leaves a head it adds the pairs to the
// workgroup's LDS keys.  Bound by its reads and
// their latency (8 waves a CU): K of 16 layers x 4080 tokens x 6 heads of 96 channels (75 MB)
// 47 us on the row kernels, 19 here (92 MB with the line halves beside a head's 192 bytes, 5.0
// TB/s); V of 16 x 4096 x 8 of 128 (134 MB) 72 -> 28 us.
template <int D>
__global__ __launch_bounds__(kTileThreads, D <= 80 ? 4 : D <= 128 ? 3 : 2) void tile_stats_kernel(Geo g, TileArgs a,
                                                                  const kvmi_layer_job* __restrict__ jobs) {
  using TG = TileGeo<D>;
  constexpr int KS = TG::KS, NC = TG::NC, PP = TG::PP;
  const kvmi_layer_job job = jobs[gridDim.y - 1 - blockIdx.y];  // see kstats_body
  const int H = g.H, S = g.S, HD = H * D;
  const int ntok = job.num_blocks * S, tok0 = blockIdx.x * a.run;
  if (tok0 >= ntok) return;
  const int tok_end = min(ntok, tok0 + a.run);
  const int parts = a.tabs == 3 ? 2 : 1, part = parts == 2 ? (int)blockIdx.z & 1 : (a.tabs >> 1);
  const bool channel = part_axis(g.flags, part) == kAxChannel;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, hl = l >> 5, r = l & 31;

  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ TileTables T;
  uint32_t* smask = reinterpret_cast<uint32_t*>(lds);
  uint32_t* lkey = reinterpret_cast<uint32_t*>(lds + a.off_tab);  // [2][HD] (channel) or [2][H] (tensor)
  uint4* tb = reinterpret_cast<uint4*>(lds + a.off_wave + wave * a.wave_bytes);
  const int nkeys = channel ? HD : H;
  tile_stage_profile(T, job.profile, H);
  tile_signs<D>(smask, job.signs, H);
  for (int i = threadIdx.x; i < nkeys; i += kTileThreads) {
    lkey[i] = 0xffffffffu;
    lkey[nkeys + i] = 0u;
  }
  __syncthreads();
  tile_positions(T, H);
  __syncthreads();

  uint4 bp[2], bn[2];  // B operands: column n = lane % 32 is channel 32 c + n of its tile
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    uint32_t w[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      w[p] = 0;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int e = 16 * kt + 8 * hl + 2 * p + s;
        w[p] |= (uint32_t)((__builtin_popcount(r & e) & 1) ? 0xBF80u : 0x3F80u) << (16 * s);
      }
    }
    bp[kt] = make_uint4(w[0], w[1], w[2], w[3]);
    bn[kt] = xor4(bp[kt], make_uint4(0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u));
  }
  const uint16_t* pool = reinterpret_cast<const uint16_t*>(job.pool) + (part ? job.pool_part_stride : 0);
  const int nk = (tok_end - tok0 + kStatTok - 1) / kStatTok, items = nk * H;
  const int waves = kTileWaves * (int)gridDim.z / parts, w = kTileWaves * ((int)blockIdx.z / parts) + wave;
  const int first = w * items / waves, end = (w + 1) * items / waves;
  // Row r's token index in the pool goes through LDS to the lanes that load the row; the
  // block ids of a tile are loaded one tile earlier than its rows.
  int* ptok = reinterpret_cast<int*>(tb + TG::kBuf);
  auto token = [&](int n) { return min(tok0 + kStatTok * (n % nk) + r, tok_end - 1); };
  auto block_id = [&](int n) { return gld(job.block_ids + tile_block_of(token(n), a)); };
  int id = 0;
  auto fetch = [&](int n, uint4 (&x)[KS]) {
    const int t = token(n);
    ptok[r] = id * S + (t - tile_block_of(t, a) * S);  // both lane halves: the same value
    id = block_id(min(n + 1, end - 1));
    const uint16_t* base = pool + (int64_t)(n / nk) * D;
#pragma unroll
    for (int v = 0; v < KS; ++v)
      x[v] = gld(reinterpret_cast<const uint4*>(base + (int64_t)ptok[tile_row_of<D>(v, l)] * HD) +
                 tile_col_of<D>(v, l));
  };
  float mn[NC], mx[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) mn[c] = __builtin_inff(), mx[c] = -__builtin_inff();
  auto take = [&](int n, uint4 (&x)[KS]) {
    const int h = n / nk;
#pragma unroll
    for (int v = 0; v < KS; ++v) pin(x[v]);
    uint4 y[2 * NC];
#pragma unroll
    for (int gi = 0; gi < TG::NG; ++gi) {
#pragma unroll
      for (int v = 0; v < TG::KG; ++v) tb[tile_slot_of<D>(v, l)] = x[gi * TG::KG + v];
#pragma unroll
      for (int s = 0; s < TG::KG; ++s) y[gi * TG::KG + s] = tb[r * PP + 2 * s + hl];
    }
    fetch(min(n + 1, end - 1), x);  // the next tile (at the end this one again)
    const uint4* sm = reinterpret_cast<const uint4*>(smask + h * (D / 2 + 4)) + hl;
#pragma unroll
    for (int s = 0; s < KS; ++s) y[s] = xor4(y[s], sm[2 * s]);
    tile_each<NC>([&](auto cpc) {
      constexpr int cp = decltype(cpc)::value;
      const f32x16 acc = tile_transform<D, cp>(y, bp, bn, [](uint4 A, uint4 B, f32x16 c) { return mfma(B, A, c); });
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        mn[cp] = fminf(mn[cp], fminf(acc[i], acc[i + 1]));
        mx[cp] = fmaxf(mx[cp], fmaxf(acc[i], acc[i + 1]));
      }
      chunk_fence();
    });
    if (n + 1 < end && (n + 1) / nk == h) return;  // the next tile is this head's
    float amn = __builtin_inff(), amx = -__builtin_inff();
    tile_each<NC>([&](auto cpc) {
      constexpr int cp = decltype(cpc)::value;
      constexpr float sc = kTileScale<D, cp>;
      const float a0 = halves_min(mn[cp]) * sc, b0 = halves_max(mx[cp]) * sc;
      mn[cp] = __builtin_inff(), mx[cp] = -__builtin_inff();
      if (channel) {
        // a 16-channel tail: columns 16 .. 31 are copies of columns 0 .. 15
        const int f = h * D + 32 * cp + (TG::kTail && cp == NC - 1 ? (r & 15) : r);
        if (hl == 0) atomicMin(&lkey[f], f2key(a0));
        else atomicMax(&lkey[HD + f], f2key(b0));
      } else {
        amn = fminf(amn, a0);
        amx = fmaxf(amx, b0);
      }
    });
    if (channel) return;
#pragma unroll
    for (int o = 16; o >= 1; o >>= 1) {
      amn = fminf(amn, __shfl_xor(amn, o, 64));
      amx = fmaxf(amx, __shfl_xor(amx, o, 64));
    }
    if (l == 0) {
      const int grp = T.prof[part][2][T.pos[part][h]];
      atomicMin(&lkey[grp], f2key(amn));
      atomicMax(&lkey[nkeys + grp], f2key(amx));
    }
  };
  if (first < end) {
    uint4 x[KS];
    id = block_id(first);
    fetch(first, x);
    for (int n = first; n < end; ++n) take(n, x);
  }
  __syncthreads();
  uint32_t* keys = job.kstats + part * 2 * HD;
  for (int i = threadIdx.x; i < nkeys; i += kTileThreads) {
    const uint32_t a0 = lkey[i], b0 = lkey[nkeys + i];
    if (a0 != 0xffffffffu) atomicMin(&keys[i], a0);
    if (b0 != 0u) atomicMax(&keys[HD + i], b0);
  }
}

// Without the transform a token's H D values are plain columns: a thread keeps 8 channels
// and walks the tokens of the run, kPlainAhead loads in flight (K of 16 layers x 4096 tokens
// x 8 heads of 128, 134 MB: 42 us on the quad kernels, 29 here, 4.7 TB/s; with the caches' rows
// still in the last-level cache 29 and 32).
constexpr int kPlainAhead = 4;
__global__ __launch_bounds__(kTileThreads) void tile_plain_stats_kernel(Geo g, TileArgs a,
                                                                        const kvmi_layer_job* __restrict__ jobs) {
  const kvmi_layer_job job = jobs[gridDim.y - 1 - blockIdx.y];
  const int H = g.H, S = g.S, D = g.D, HD = H * D, PT = HD / 8;  // pieces of a token
  const int ntok = job.num_blocks * S, tok0 = blockIdx.x * a.run;
  if (tok0 >= ntok) return;
  const int tok_end = min(ntok, tok0 + a.run);
  const int part = (a.tabs == 3) ? (int)blockIdx.z : (a.tabs >> 1);
  const bool channel = part_axis(g.flags, part) == kAxChannel;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ TileTables T;
  uint32_t* lkey = reinterpret_cast<uint32_t*>(lds);
  const int nkeys = channel ? HD : H;
  tile_stage_profile(T, job.profile, H);
  for (int i = threadIdx.x; i < nkeys; i += kTileThreads) {
    lkey[i] = 0xffffffffu;
    lkey[nkeys + i] = 0u;
  }
  __syncthreads();
  tile_positions(T, H);
  __syncthreads();
  const int lanes = kTileThreads / PT;  // tokens the workgroup reads at once (PT <= kTileThreads)
  const int c = threadIdx.x % PT, w = threadIdx.x / PT;
  const uint16_t* pool = reinterpret_cast<const uint16_t*>(job.pool) + (part ? job.pool_part_stride : 0);
  float mn[8], mx[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) mn[i] = __builtin_inff(), mx[i] = -__builtin_inff();
  if (w < lanes) {
    for (int t0 = tok0 + w; t0 < tok_end; t0 += kPlainAhead * lanes) {
      uint4 x[kPlainAhead];
#pragma unroll
      for (int u = 0; u < kPlainAhead; ++u) {
        const int t = min(t0 + u * lanes, tok_end - 1);
        const int b = tile_block_of(t, a);
        const int64_t row = (int64_t)gld(job.block_ids + b) * S + (t - b * S);
        x[u] = gld(reinterpret_cast<const uint4*>(pool + row * HD) + c);
      }
#pragma unroll
      for (int u = 0; u < kPlainAhead; u += 2) {
        const uint32_t p[4] = {x[u].x, x[u].y, x[u].z, x[u].w}, q[4] = {x[u + 1].x, x[u + 1].y, x[u + 1].z, x[u + 1].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          mn[2 * i] = fminf(mn[2 * i], fminf(bf_lo(p[i]), bf_lo(q[i])));
          mx[2 * i] = fmaxf(mx[2 * i], fmaxf(bf_lo(p[i]), bf_lo(q[i])));
          mn[2 * i + 1] = fminf(mn[2 * i + 1], fminf(bf_hi(p[i]), bf_hi(q[i])));
          mx[2 * i + 1] = fmaxf(mx[2 * i + 1], fmaxf(bf_hi(p[i]), bf_hi(q[i])));
        }
      }
    }
    if (tok0 + w < tok_end) {
      if (channel) {
        // slot (i + piece) % 8 of the piece, so that neighbouring lanes use other banks
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int s = 8 * c + ((i + c) & 7);
          atomicMin(&lkey[s], f2key(mn[i]));
          atomicMax(&lkey[HD + s], f2key(mx[i]));
        }
      } else {
        float lo = mn[0], hi = mx[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) lo = fminf(lo, mn[i]), hi = fmaxf(hi, mx[i]);
        const int grp = T.prof[part][2][T.pos[part][8 * c / D]];
        atomicMin(&lkey[grp], f2key(lo));
        atomicMax(&lkey[nkeys + grp], f2key(hi));
      }
    }
  }
  __syncthreads();
  uint32_t* keys = job.kstats + part * 2 * HD;
  for (int i = threadIdx.x; i < nkeys; i += kTileThreads) {
    const int s = channel ? (i & ~7) + ((i + (i >> 3)) & 7) : i;
    const uint32_t a0 = lkey[s], b0 = lkey[nkeys + s];
    if (a0 != 0xffffffffu) atomicMin(&keys[i], a0);
    if (b0 != 0u) atomicMax(&keys[HD + i], b0);
  }
}

constexpr int round16(int x) { return (x + 15) & ~15; }

int tab_mask(const Geo& g) {
  return (part_axis(g.flags, 0) != kAxToken ? 1 : 0) | (part_axis(g.flags, 1) != kAxToken ? 2 : 0);
}

// Bytes of a wave's tile buffer (TileGeo::kBuf).
int buffer_bytes(int D) { return kTok * ((D % 64 ? D / 8 : 8) + 1) * 16; }

// Everything of a launch shape but its run and super-tile; `nt` tiles of image per wave.
TileArgs shape(const Geo& g, int nt) {
  TileArgs a{};
  const bool tr = !(g.flags & KVMI_F_NO_TRANSFORM), native = g.flags & KVMI_F_NATIVE_LAYOUT;
  const int RB = g.D * g.bits / 8;
  a.T = kTok / g.H < g.S ? kTok / g.H : g.S;
  a.ST = a.T * nt;
  a.magic = g.S == 1 ? 0u : (uint32_t)((1ull << 32) / (unsigned)g.S + 1ull);
  a.tabs = tab_mask(g);
  a.runs = native ? 1 : g.H;
  // 16 bytes behind each run: its banks differ from the next one's, and the last symbols of
  // a row may be read as a whole dword or two
  a.pitch = round16(a.ST * RB * (native ? g.H : 1)) + 16;
  a.off_tab = tr ? g.H * (g.D / 2 + 4) * 4 : 0;
  a.off_wave = a.off_tab + ((a.tabs & 1) + (a.tabs >> 1)) * g.H * (g.D + 4) * 8;
  a.wave_bytes = buffer_bytes(g.D) + a.runs * a.pitch;
  return a;
}
int lds_bytes(const TileArgs& a) { return a.off_wave + kTileWaves * a.wave_bytes; }
int slots(const Geo& g, const TileArgs& a) {
  const int RB = g.D * g.bits / 8;
  return a.runs * ((a.ST * RB * (a.runs == 1 && (g.flags & KVMI_F_NATIVE_LAYOUT) ? g.H : 1) + 15) / 16);
}

constexpr int kStaticLds = 1024;                  // TileTables and the like, rounded up
constexpr int kMaxLds = 80 * 1024 - kStaticLds;   // two workgroups a CU
// A wave's image grows, tile by tile, until a head's run in the stream is kRunBytes long, or the
// image has more slots than a wave of decode holds (max_slots; that ends 6 heads of 96 at 480
// bytes and 8 of 128 at 512, 4 heads of 64 go to 768), or a wave would be left without a
// super-tile.  One tile an image against the rule, at 16 layers and 4 bits (encode / decode us):
// 4080 tokens x 6 of 96: 240 bytes 57.9 / 50.5, 480 bytes 55.6 / 45.4; 4096 x 12 of 192: 192
// bytes 239 / 226, 576 bytes 229 / 199; K per token and V per channel 4096 x 8 of 128: 256 bytes
// 85.4 / 68.5, 512 bytes 82.0 / 64.3; 8192 x 4 of 64: 256 bytes 46.9 / 40.7, 768 bytes 44.4 / 34.3
// (1024 bytes 41.4 / 37.5).
constexpr int kRunBytes = 720;
constexpr int kTileRounds = 3;  // workgroups per resident slot: 1, 2, 4 and 6 within 5 %
// 16-byte slots of an image: 64 * kPackedRegs of kvmi_tile_dec.hip
int max_slots(const Geo& g) { return g.D <= 128 ? 256 : 512; }

template <int D>
int launch_stats(const Geo& g, const TileArgs& a, dim3 grid, const kvmi_layer_job* jobs, size_t lds, hipStream_t st) {
  hipLaunchKernelGGL(tile_stats_kernel<D>, grid, dim3(kTileThreads), lds, st, g, a, jobs);
  return hipGetLastError() == hipSuccess ? KVMI_OK : KVMI_ELAUNCH;
}

}  // namespace

int tile_cus() {
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      return 256;
    return n;
  }();
  return cus;
}

namespace {

// What the kernels can do: their head sizes, 32-bit offsets, and the LDS of a workgroup.
// Decode needs two workgroups a CU (8 layers x 1024 tokens of 10 heads of 256, both parts by
// channel: one 73 us, the row kernels 48); compress still gains with one (4096 tokens 568 -> 413).
bool tile_eligible(const Geo& g, int32_t max_blocks, bool decode) {
  if (g.flags & (KVMI_F_VALU_FWHT | KVMI_F_ROW_FWHT | kPairedHeads)) return false;
  if (g.H > kTileMaxH) return false;
  switch (g.D) {
    case 64: case 80: case 96: case 112: case 128: case 160: case 192: case 224: case 256: break;
    default: return false;
  }
  const int64_t tokens = (int64_t)max_blocks * g.S;
  if (tokens >= (1ll << 30) || tokens * g.S >= (1ll << 32)) return false;  // the division by S
  if (tokens * g.H * g.D * g.bits / 8 >= (1ll << 32)) return false;        // 32-bit offsets in a part's stream
  if ((g.flags & KVMI_F_NO_TRANSFORM) && g.H * g.D / 8 > kTileThreads) return false;
  const TileArgs a = shape(g, 1);
  return lds_bytes(a) <= kMaxLds + (decode ? 0 : kStaticLds) && slots(g, a) <= max_slots(g);
}

// Whether they are the faster ones.  A tile of few rows (small blocks, awkward head counts)
// costs what a full one does, and what it competes with differs: the quad kernels are about
// twice as fast as the row kernels, and the row kernels spend next_pow2(D) channels on D.  The
// rule looks at the geometry alone: with the call's length in it, a request's bytes could
// depend on the batch it is in.  Compress / decompress (us) of 8 layers x 8192 tokens, the other
// kernels -> tiles, and the rows of a tile:
//   quad  8 x 128, S = 1:  8 rows 296 -> 267 / 160 -> 181     S = 2: 16 rows 295 -> 175 / 160 -> 111
//         4 x 128, S = 2:  8 rows 136 -> 153 /  67 -> 103     S = 4: 16 rows 136 ->  96 /  66 ->  61
//         1 x 128, S = 8:  8 rows  42 ->  48 /  19 ->  33    S = 16: 16 rows  42 ->  35 /  19 ->  22
//         8 x 64,  S = 2: 16 rows 131 ->  90 /  51 ->  58; 1024 tokens, 16 x 64, S = 1: 1.18 times the time
//   rows  5 x 128, S = 1:  5 rows 279 -> 279 / 119 -> 197     S = 2: 10 rows 280 -> 159 / 118 -> 109
//        10 x 128, S = 1: 10 rows 613 -> 304 / 279 -> 211, but 1024 tokens decompress 1.0 - 1.3 times the time
//         8 x 96,  S = 1:  8 rows 433 -> 204 / 168 -> 137    12 x 96, S = 1: 12 rows 759 -> 254 / 296 -> 190
// Short calls of few large heads stay slower than on the other kernels, however full the tiles
// are: the latency of one tile.  Up to about 1000 tokens of 1 - 5 heads decompress takes 1 - 3 us
// longer from 160 channels on (1 x 224 at 528 x 4: 7.9 -> 12.4), compress 3 - 8 us at 256 (5 heads
// at 128 x 8: 22 -> 30).
bool tile_faster(const Geo& g, bool decode) {
  const int rows = shape(g, 1).T * g.H;
  if (decode && (g.flags & KVMI_F_NO_TRANSFORM) && g.H > 16) return false;  // short image runs: 1024 x 8 x 32 of 64 26 -> 31 us
  if (quad_eligible(g)) return decode ? rows >= 20 : rows * g.D >= 16 * 128;
  const bool waste = 4 * next_pow2(g.D) >= 5 * g.D;  // of the row kernels: 80, 96, 160 and 192 channels
  // 12 rows: only at 4 bits, which has code of its own (1770 x 8 of 12 x 96 at 5 bits 50 -> 74 us), and
  // not with one token a tile beyond 16 heads (960 x 8 of 17 x 128 45 -> 49)
  if (decode) return rows >= 20 || (waste && g.bits == 4 && g.H <= 16 && rows >= 12);
  return rows >= (waste ? 8 : 10);
}

}  // namespace

bool tile_serves(const Geo& g, int32_t max_blocks, bool decode) {
  return tile_eligible(g, max_blocks, decode) && tile_faster(g, decode);
}

TileArgs tile_plan(const Geo& g, int32_t max_blocks, int32_t num_jobs, int occ) {
  const int64_t tokens = (int64_t)max_blocks * g.S;
  const int T = shape(g, 1).T, RB = g.D * g.bits / 8;
  const int64_t tiles = (tokens + T - 1) / T * num_jobs;
  // workgroups resident at once: by registers (occ waves a SIMD) and by LDS
  auto resident = [&](const TileArgs& a) {
    const int by_lds = 160 * 1024 / (lds_bytes(a) + kStaticLds);
    return (int64_t)tile_cus() * (occ < by_lds ? occ : by_lds);
  };
  int nt = 1;
  for (int k = 2; k <= 16 && (nt * T) * RB < kRunBytes; ++k) {
    const TileArgs b = shape(g, k);
    if (slots(g, b) > max_slots(g) || lds_bytes(b) > kMaxLds ||
        tiles / k < resident(b) * kTileWaves)
      break;
    nt = k;
  }
  TileArgs a = shape(g, nt);
  const int64_t unit = (int64_t)kTileWaves * a.ST, want = resident(a) * kTileRounds;  // workgroups
  int64_t run = (tokens * num_jobs + want - 1) / want;
  run = (run + unit - 1) / unit * unit;
  const int64_t most = (tokens + unit - 1) / unit * unit;
  a.run = (int)(run < unit ? unit : run > most ? most : run);
  // few tiles: K and V in workgroups of their own, half the serial work of a wave
  a.parts = (tokens + a.run - 1) / a.run * num_jobs * 2 <= resident(a) ? 1 : 2;
  return a;
}

void tile_shape(const Geo& g, int32_t num_jobs, int32_t max_blocks, int32_t (&out)[4]) {
  const TileArgs a = tile_plan(g, max_blocks, num_jobs, tile_occ(g.D));
  out[0] = a.T, out[1] = a.ST / a.T, out[2] = a.run, out[3] = a.parts;
}

int tile_kstats(const Geo& g, const kvmi_layer_job* jobs, int32_t num_jobs, int32_t max_blocks, int32_t*,
                hipStream_t st) {
  TileArgs a = shape(g, 1);
  if (!a.tabs) return KVMI_OK;  // both parts take their statistics per token, in encode
  const bool tr = !(g.flags & KVMI_F_NO_TRANSFORM);
  const unsigned parts = a.tabs == 3 ? 2 : 1;
  const int64_t tokens = (int64_t)max_blocks * g.S;
  // workgroups a CU, at least one tile a wave: with the transform 2 (fewer table set-ups and
  // key atomics; 3 and 4: 7 and 20 % slower on 16 layers x 4096 tokens, 3 % either way on 32 x
  // 8192), without 6
  const int64_t want = (int64_t)tile_cus() * (tr ? 2 : 6);
  int64_t run = (tokens * num_jobs * parts + want - 1) / want;
  const int64_t unit = tr ? kStatTok : 1, least = tr ? kStatTok * ((kTileWaves + g.H - 1) / g.H)
                                              : 2 * kPlainAhead * (kTileThreads / (g.H * g.D / 8));
  run = run < least ? least : (run + unit - 1) / unit * unit;
  a.run = (int)(run > tokens ? (tokens + unit - 1) / unit * unit : run);
  // a short call leaves the chip idle and a wave walks several heads: more workgroups a run, down
  // to a tile a wave (8 layers x 64 tokens x 10 heads of 256: 29 -> 16 us, row kernels 16)
  const int64_t groups = (tokens + a.run - 1) / a.run * num_jobs * parts, items = (int64_t)(a.run / kStatTok) * g.H;
  int64_t share = 1;
  if (tr) share = std::max<int64_t>(1, std::min(want / groups, (items + kTileWaves - 1) / kTileWaves));
  const dim3 grid((unsigned)((tokens + a.run - 1) / a.run), (unsigned)num_jobs, (unsigned)(parts * share));
  const size_t keys = (size_t)2 * g.H * g.D * 4;
  int rc;
  if (tr) {
    a.off_wave = a.off_tab + (int)keys;
    a.wave_bytes = buffer_bytes(g.D) + kTok * 4;  // tile buffer, token indexes
    const size_t lds = (size_t)lds_bytes(a);
    switch (g.D) {
      case 64: rc = launch_stats<64>(g, a, grid, jobs, lds, st); break;
      case 80: rc = launch_stats<80>(g, a, grid, jobs, lds, st); break;
      case 96: rc = launch_stats<96>(g, a, grid, jobs, lds, st); break;
      case 112: rc = launch_stats<112>(g, a, grid, jobs, lds, st); break;
      case 128: rc = launch_stats<128>(g, a, grid, jobs, lds, st); break;
      case 160: rc = launch_stats<160>(g, a, grid, jobs, lds, st); break;
      case 192: rc = launch_stats<192>(g, a, grid, jobs, lds, st); break;
      case 224: rc = launch_stats<224>(g, a, grid, jobs, lds, st); break;
      default: rc = launch_stats<256>(g, a, grid, jobs, lds, st); break;
    }
  } else {
    hipLaunchKernelGGL(tile_plain_stats_kernel, grid, dim3(kTileThreads), keys, st, g, a, jobs);
    rc = hipGetLastError() == hipSuccess ? KVMI_OK : KVMI_ELAUNCH;
  }
  if (rc) return rc;
  return rows_finalize(g, jobs, num_jobs, st);
}

}  // namespace kvmi
