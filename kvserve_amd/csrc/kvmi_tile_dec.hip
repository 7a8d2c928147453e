// Decode pass of the wave-tile kernels (kvmi_tile.hpp): unpack, dequantize on any axis,
// inverse transform, scatter into the paged caches.
//
// Bound by its writes in long requests, which reach the rate of a device copy (32 layers x 8192
// tokens x 8 heads of 128 channels without transform 1.34 GB in 0.22 ms); in shorter ones by vector
// issue (half to two thirds of the busy time), trips to memory (half of a wave's time) and a partly
// filled last round (profiles/case_kernels.md).  Against the row kernels that ran these calls
// before: 16 layers x 4080 tokens x 6 heads of 96 channels 141 -> 47 us (192 MB, 4.1 TB/s), 16 x
// 4096 x 8 of 128 with K per token and V per channel 173 -> 74, without the transform (quad kernels
// before) 143 -> 63 us (342 MB, 5.4 TB/s).
#include "kvmi_tile.hpp"

namespace kvmi {
namespace {

// 16-byte slots a lane holds of the next image
template <int D>
constexpr int kPackedRegs = D <= 128 ? 4 : 8;

// The 8 symbols at `p` (BITS bytes, any alignment) as floats.
template <int BITS>
__device__ __forceinline__ void unpack8(const uint8_t* p, float (&s)[8]) {
  if constexpr (BITS <= 4) {
    const uint32_t w = BITS == 4 ? *reinterpret_cast<const uint32_t*>(p) : reinterpret_cast<const Word1*>(p)->v;
    if constexpr (BITS == 4) {
      const uint32_t lo = barrier_u(w & 0x0F0F0F0Fu), hi = barrier_u((w >> 4) & 0x0F0F0F0Fu);
      s[0] = ubyte<0>(lo), s[1] = ubyte<0>(hi), s[2] = ubyte<1>(lo), s[3] = ubyte<1>(hi);
      s[4] = ubyte<2>(lo), s[5] = ubyte<2>(hi), s[6] = ubyte<3>(lo), s[7] = ubyte<3>(hi);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) s[j] = (float)((w >> (j * BITS)) & ((1u << BITS) - 1u));
    }
  } else {
    const Word2 v = *reinterpret_cast<const Word2*>(p);
    if constexpr (BITS == 8) {
      s[0] = ubyte<0>(v.a), s[1] = ubyte<1>(v.a), s[2] = ubyte<2>(v.a), s[3] = ubyte<3>(v.a);
      s[4] = ubyte<0>(v.b), s[5] = ubyte<1>(v.b), s[6] = ubyte<2>(v.b), s[7] = ubyte<3>(v.b);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int bit = j * BITS;
        uint32_t x = bit < 32 ? v.a >> (bit & 31) : v.b >> (bit & 31);
        if (bit < 32 && bit + BITS > 32) x |= v.b << (32 - bit);
        s[j] = (float)(x & ((1u << BITS) - 1u));
      }
    }
  }
}
// BITS 0: the width is a run-time value.
template <int BITS>
__device__ __forceinline__ void unpack8_bits(int bits, const uint8_t* p, float (&s)[8]) {
  if constexpr (BITS != 0) return unpack8<BITS>(p, s);
  switch (bits) {  // uniform
    case 3: return unpack8<3>(p, s);
    case 8: return unpack8<8>(p, s);
    case 2: return unpack8<2>(p, s);
    case 6: return unpack8<6>(p, s);
    case 5: return unpack8<5>(p, s);
    case 7: return unpack8<7>(p, s);
    default: return unpack8<1>(p, s);
  }
}

template <int D, bool TR, int BITS>
__global__ __launch_bounds__(kTileThreads, tile_occ(D)) void tile_decode_kernel(Geo g, TileArgs a,
                                                                               const kvmi_layer_job* __restrict__ jobs,
                                                                               int32_t* __restrict__ err) {
  using TG = TileGeo<D>;
  constexpr int KS = TG::KS, NC = TG::NC, PP = TG::PP;
  const kvmi_layer_job job = jobs[blockIdx.y];
  const int H = g.H, bits = BITS ? BITS : g.bits, RB = D * bits / 8;
  const int ntok = job.num_blocks * g.S;
  const int tok0 = blockIdx.x * a.run;
  if (tok0 >= ntok) return;
  const int tok_end = min(ntok, tok0 + a.run);
  const int part0 = a.parts == 1 ? (int)blockIdx.z : 0, part1 = part0 + a.parts;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, hl = l >> 5, r = l & 31;

  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ TileTables T;
  uint32_t* smask = reinterpret_cast<uint32_t*>(lds);
  float2* kc = reinterpret_cast<float2*>(lds + a.off_tab);
  uint4* tb = reinterpret_cast<uint4*>(lds + a.off_wave + wave * a.wave_bytes);
  uint8_t* img = reinterpret_cast<uint8_t*>(tb + TG::kBuf);
  const bool native = g.flags & KVMI_F_NATIVE_LAYOUT;

  // Packed image of (part, super-tile at `tok`).  Runs under 16 bytes (a few tokens at the
  // end of a narrow job) are read where they are used, 2 bytes at a time.
  const uint32_t stride = (uint32_t)ntok * (uint32_t)RB;  // between the runs of a part's heads
  auto run_bytes = [&](int tok) { return (min(tok_end, tok + a.ST) - tok) * RB * (native ? H : 1); };
  auto fetch = [&](int part, int tok, uint4 (&x)[kPackedRegs<D>]) {
    const TileSlots s = tile_slots(run_bytes(tok), a.runs);
    if (s.rl < 16) return;
    const uint8_t* base = tile_stream(job, g, part, 0, tok, ntok, RB);
#pragma unroll
    for (int u = 0; u < kPackedRegs<D>; ++u) {
      if (64 * u >= s.count) break;
      int j, off;
      tile_slot(s, min(64 * u + l, s.count - 1), j, off);
      x[u] = ld16u(base + ((uint32_t)j * stride + (uint32_t)off));
    }
  };
  auto put = [&](int part, int tok, const uint4 (&x)[kPackedRegs<D>]) {
    const TileSlots s = tile_slots(run_bytes(tok), a.runs);
    if (s.rl < 16) {
      const uint8_t* base = tile_stream(job, g, part, 0, tok, ntok, RB);
      const int ns = s.rl >> 1;
      for (int q = l; q < a.runs * ns; q += 64) {
        const int j = q / ns, off = 2 * (q - j * ns);
        *reinterpret_cast<u16any*>(img + j * a.pitch + off) =
            gld(reinterpret_cast<const uint16_t*>(base + ((uint32_t)j * stride + (uint32_t)off)));
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < kPackedRegs<D>; ++u) {
      if (64 * u >= s.count) break;
      int j, off;
      tile_slot(s, min(64 * u + l, s.count - 1), j, off);
      Bytes16* d = reinterpret_cast<Bytes16*>(img + (int)__umul24(j, a.pitch) + off);
      d->x = x[u].x;
      d->y = x[u].y;
      d->z = x[u].z;
      d->w = x[u].w;
    }
  };
  // The stream is as long as its header says, so nothing of it is read before the header
  // matches: every wave checks for itself, while the loads of the first tables are in flight.
  // The first image's loads are then in flight during the rest of the table set-up.
  const bool ok = (g.flags & KVMI_F_NO_HEADER) || header_matches(job.stream, bits, job.chunk_symbols);
  tile_stage_profile(T, job.profile, H);
  if (TR) tile_signs<D>(smask, job.signs, H);
  if (!ok) {  // the same for the whole workgroup
    if (threadIdx.x == 0 && blockIdx.x == 0 && part0 == 0) atomicOr(err, KVMI_ERR_BAD_HEADER);
    return;
  }
  const int step = kTileWaves * a.ST;
  int st = tok0 + wave * a.ST;
  uint4 pk[kPackedRegs<D>];
  if (st < tok_end) fetch(part0, st, pk);
  __syncthreads();
  tile_positions(T, H);
  const int tab1 = (a.tabs & 1) ? H * (D + 4) : 0;
  if ((a.tabs & 1) && part0 == 0) tile_consts<D, false>(kc, T, g, job.kmeta, 0);
  if ((a.tabs & 2) && part1 == 2) tile_consts<D, false>(kc + tab1, T, g, job.vmeta, 1);
  __syncthreads();
  if (st >= tok_end) return;

  const int h = r % H, tt = min(r / H, a.T - 1);  // rows past the tile's tokens repeat its last token
  const int jk = T.pos[0][h], jv = T.pos[1][h];
  const int grpk = T.prof[0][2][jk], grpv = T.prof[1][2][jv];
  uint4 hp[2], hn[2];
  if (TR) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      hp[kt] = hadamard_tile_d(kt, false);
      hn[kt] = hadamard_tile_d(kt, true);
    }
  }

  for (; st < tok_end; st += step) {
    const int ste = min(tok_end, st + a.ST);
#pragma unroll 1  // one copy of the section's code for both parts
    for (int part = part0; part < part1; ++part) {
      const bool table = (a.tabs >> part) & 1;
      const int jpos = part ? jv : jk, grp = part ? grpv : grpk;
      put(part, st, pk);
      if (part + 1 < part1)
        fetch(part + 1, st, pk);
      else if (st + step < tok_end)
        fetch(part0, st + step, pk);
      const uint16_t* meta = part ? job.vmeta : job.kmeta;
      for (int ta = st; ta < ste; ta += a.T) {
        const int nt = min(a.T, ste - ta);
        const uint8_t* in = img + (native ? ((ta - st + tt) * H + jpos) * RB
                                          : jpos * a.pitch + (ta - st + tt) * RB);
        float rmn = 0.f, rsc = 0.f;
        if (!table) {
          const int tok = min(ta + tt, ste - 1);
          rmn = bf16_to_f32(gld(meta + (int64_t)grp * ntok + tok));
          rsc = bf16_to_f32(gld(meta + (int64_t)(g.G + grp) * ntok + tok));
        }
        const float2* kd = kc + opaque((part ? tab1 : 0) + h * (D + 4) + 8 * hl);
        uint4 x[2 * NC];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          float sy[8];
          unpack8_bits<BITS>(bits, in + (2 * s + hl) * bits, sy);
          uint32_t w[4];
          if (table) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
              const float4 c = *reinterpret_cast<const float4*>(kd + 16 * s + 2 * p);
              // a product that is infinite stays in its own channel (see tile_diff)
              w[p] = pack_bf16x2(rbf(sy[2 * p] * c.y) + c.x, rbf(sy[2 * p + 1] * c.w) + c.z);
            }
          } else {
#pragma unroll
            for (int p = 0; p < 4; ++p) w[p] = pack_bf16x2(rbf(sy[2 * p] * rsc) + rmn, rbf(sy[2 * p + 1] * rsc) + rmn);
          }
          x[s] = make_uint4(w[0], w[1], w[2], w[3]);
        }
        uint4* row = tb + r * PP;
        const TileRows t = tile_rows<D>(job, g, a, part, ta, nt);
        if constexpr (TR) {
          chunk_fence();
          const uint4* sm = reinterpret_cast<const uint4*>(smask + opaque(h * (D / 2 + 4)));
          tile_each<NC>([&](auto cpc) {
            constexpr int cp = decltype(cpc)::value, gi = TG::kHalves ? cp / 2 : 0;
            constexpr float sc = kTileScale<D, cp>;
            const f32x16 acc = tile_transform<D, cp>(x, hp, hn, [](uint4 A, uint4 B, f32x16 c) { return mfma(A, B, c); });
            uint32_t w[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) w[i] = pack_bf16x2(acc[2 * i] * sc, acc[2 * i + 1] * sc);
            // a 16-channel tail: both lane halves hold it and write the same bytes
            const int at = 4 * cp + (TG::kTail && cp == NC - 1 ? 0 : 2 * hl);
            row[at - gi * TG::PG] = xor4(make_uint4(w[0], w[1], w[2], w[3]), sm[at]);
            row[at + 1 - gi * TG::PG] = xor4(make_uint4(w[4], w[5], w[6], w[7]), sm[at + 1]);
            if constexpr (TG::kHalves && cp % 2 == 1) tile_store<D>(t, gi, l, tb);
            chunk_fence();
          });
          if constexpr (!TG::kHalves) tile_store<D>(t, 0, l, tb);
        } else {
#pragma unroll
          for (int gi = 0; gi < TG::NG; ++gi) {
#pragma unroll
            for (int s = 0; s < TG::KG; ++s) row[2 * s + hl] = x[gi * TG::KG + s];
            tile_store<D>(t, gi, l, tb);
          }
        }
      }
    }
  }
}

template <int D, bool TR, int BITS>
int launch_b(const Geo& g, const kvmi_layer_job* jobs, int32_t nj, int32_t mb, int32_t* err, hipStream_t st) {
  const TileArgs a = tile_plan(g, mb, nj, tile_occ(D));
  const unsigned gx = (unsigned)(((int64_t)mb * g.S + a.run - 1) / a.run);
  const size_t lds = (size_t)a.off_wave + (size_t)kTileWaves * a.wave_bytes;
  hipLaunchKernelGGL((tile_decode_kernel<D, TR, BITS>), dim3(gx, (unsigned)nj, a.parts == 1 ? 2 : 1), dim3(kTileThreads),
                     lds, st, g, a, jobs, err);
  return hipGetLastError() == hipSuccess ? KVMI_OK : KVMI_ELAUNCH;
}
template <int D, bool TR>
int launch_d(const Geo& g, const kvmi_layer_job* jobs, int32_t nj, int32_t mb, int32_t* err, hipStream_t st) {
  return g.bits == 4 ? launch_b<D, TR, 4>(g, jobs, nj, mb, err, st) : launch_b<D, TR, 0>(g, jobs, nj, mb, err, st);
}

}  // namespace

int tile_decode(const Geo& g, const kvmi_layer_job* jobs, int32_t nj, int32_t mb, int32_t* err, hipStream_t st) {
  const bool tr = !(g.flags & KVMI_F_NO_TRANSFORM);
#define KVMI_TILE_D(D) \
  case D: return tr ? launch_d<D, true>(g, jobs, nj, mb, err, st) : launch_d<D, false>(g, jobs, nj, mb, err, st);
  switch (g.D) {
    KVMI_TILE_D(64)
    KVMI_TILE_D(80)
    KVMI_TILE_D(96)
    KVMI_TILE_D(112)
    KVMI_TILE_D(128)
    KVMI_TILE_D(160)
    KVMI_TILE_D(192)
    KVMI_TILE_D(224)
    KVMI_TILE_D(256)
    default: return KVMI_EINVAL;
  }
#undef KVMI_TILE_D
}

}  // namespace kvmi
