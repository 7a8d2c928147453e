// Encode pass of the wave-tile kernels (kvmi_tile.hpp): gather, transform, quantize on any
// axis, bitpack.
//
// Bound by vector issue (71 % of the time its CUs are busy, conversions counted once though they
// take two slots) and by the trips to memory behind it (a wave waits for 39 % of its time at 12
// waves a CU); it reads and writes what it must, 150 + 40 MB of 16 layers x 4080 tokens x 6
// heads of 96 channels at 3.3 TB/s (profiles/case_kernels.md).  Against the row kernels that ran
// these calls before: that one 259 -> 57 us, 16 x 4096 x 8 of 128 with K per token and V per
// channel 283 -> 87, without the transform (quad kernels before) 200 -> 74 us (343 MB, 4.6 TB/s).
#include "kvmi_tile.hpp"

namespace kvmi {
namespace {

// Symbols of 16 quantized values, packed to BITS bits into 2 * BITS bytes at `dst` (LDS).
template <int BITS>
__device__ __forceinline__ void pack16(const float (&q)[16], uint8_t* dst, bool keep, uint32_t& over) {
  LanePack<16, BITS> pk;
  pk.clear();
  pack_chunk<16, BITS>(q, 0, pk, over);
  if (!keep) return;
  if constexpr (BITS == 8) {
    *reinterpret_cast<uint4*>(dst) = make_uint4(pk.w[0], pk.w[1], pk.w[2], pk.w[3]);
  } else if constexpr (BITS == 4) {
    *reinterpret_cast<uint2*>(dst) = make_uint2(pk.w[0], pk.w[1]);
  } else if constexpr (BITS == 2) {
    *reinterpret_cast<uint32_t*>(dst) = pk.w[0];
  } else if constexpr (BITS == 6) {
#pragma unroll
    for (int i = 0; i < 3; ++i) reinterpret_cast<uint32_t*>(dst)[i] = pk.w[i];
  } else {
#pragma unroll
    for (int i = 0; i < BITS; ++i) reinterpret_cast<uint16_t*>(dst)[i] = (uint16_t)(pk.w[i / 2] >> (16 * (i & 1)));
  }
}
// BITS 0: the width is a run-time value.
template <int BITS>
__device__ __forceinline__ void pack16_bits(int bits, const float (&q)[16], uint8_t* dst, bool keep, uint32_t& over) {
  if constexpr (BITS != 0) return pack16<BITS>(q, dst, keep, over);
  switch (bits) {  // uniform
    case 3: return pack16<3>(q, dst, keep, over);
    case 8: return pack16<8>(q, dst, keep, over);
    case 2: return pack16<2>(q, dst, keep, over);
    case 6: return pack16<6>(q, dst, keep, over);
    case 5: return pack16<5>(q, dst, keep, over);
    case 7: return pack16<7>(q, dst, keep, over);
    default: return pack16<1>(q, dst, keep, over);
  }
}

// Write the image of a super-tile: run j to base + j * stride.
__device__ __forceinline__ void flush_image(const uint8_t* img, int pitch, int runs, int rl, uint8_t* base,
                                            uint32_t stride, int l) {
  if (rl >= 16) {
    const TileSlots s = tile_slots(rl, runs);
    for (int q = l; q < s.count; q += 64) {
      int j, off;
      tile_slot(s, q, j, off);
      const Bytes16* v = reinterpret_cast<const Bytes16*>(img + (int)__umul24(j, pitch) + off);
      st16u(base + ((uint32_t)j * stride + (uint32_t)off), make_uint4(v->x, v->y, v->z, v->w));
    }
  } else {
    const int ns = rl >> 1;  // rows are whole 2-byte pieces (D is a multiple of 16)
    for (int q = l; q < runs * ns; q += 64) {
      const int j = q / ns, off = 2 * (q - j * ns);
      gst(reinterpret_cast<uint16_t*>(base + ((uint32_t)j * stride + (uint32_t)off)),
          (uint16_t)*reinterpret_cast<const u16any*>(img + j * pitch + off));
    }
  }
}

// min(q, level) in one instruction (level for a NaN, as the row kernels' clamp gives).
__device__ __forceinline__ float clamp_level(float q, float lev) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(q), "v"(lev));
  return r;
}

// (bf16(m0 - lo(y)), bf16(m1 - hi(y))).  Not the dot products of rsub_rbf_pair: those multiply
// the pair's other element by 0, so that an infinity would reach its neighbour, and behind a
// transform too a sum may overflow in one channel alone.  Written out, because the compiler
// unpacks the pairs of a whole tile at once and spills (D = 128: 108 bytes a lane, K per token
// and V per channel of 16 x 4096 x 8 x 128 both ways 223 us against 201).
__device__ __forceinline__ void tile_diff(uint32_t y, float m0, float m1, float& t0, float& t1) {
  asm("v_lshlrev_b32 %0, 16, %2\n\t"
      "v_and_b32 %1, 0xffff0000, %2\n\t"
      "v_sub_f32 %0, %3, %0\n\t"
      "v_sub_f32 %1, %4, %1\n\t"
      "v_cvt_pk_bf16_f32 %0, 0, %0\n\t"
      "v_cvt_pk_bf16_f32 %1, 0, %1"
      : "=&v"(t0), "=&v"(t1)
      : "v"(y), "v"(m0), "v"(m1));
}

template <int D, bool TR, int BITS>
__global__ __launch_bounds__(kTileThreads, tile_occ(D)) void tile_encode_kernel(Geo g, TileArgs a,
                                                                               const kvmi_layer_job* __restrict__ jobs,
                                                                               int32_t* __restrict__ err) {
  using TG = TileGeo<D>;
  constexpr int KS = TG::KS, NC = TG::NC, PP = TG::PP;
  const kvmi_layer_job job = jobs[blockIdx.y];
  const int H = g.H, bits = BITS ? BITS : g.bits, RB = D * bits / 8;
  const int ntok = job.num_blocks * g.S;
  const int tok0 = blockIdx.x * a.run;
  const int part0 = a.parts == 1 ? (int)blockIdx.z : 0, part1 = part0 + a.parts;
  const bool header = threadIdx.x == 0 && part0 == 0 && blockIdx.x == 0 && job.write_header && !(g.flags & KVMI_F_NO_HEADER);
  if (header) write_stream_header(job.stream, bits, job.chunk_symbols);
  if (tok0 >= ntok) return;
  const int tok_end = min(ntok, tok0 + a.run);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, hl = l >> 5, r = l & 31;

  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ TileTables T;
  uint32_t* smask = reinterpret_cast<uint32_t*>(lds);
  float2* kc = reinterpret_cast<float2*>(lds + a.off_tab);
  uint4* tb = reinterpret_cast<uint4*>(lds + a.off_wave + wave * a.wave_bytes);
  uint8_t* img = reinterpret_cast<uint8_t*>(tb + TG::kBuf);
  // the first tile's loads are in flight during the table set-up
  const int step = kTileWaves * a.ST;
  int st = tok0 + wave * a.ST;
  uint4 pf[KS];
  if (st < tok_end) tile_load<D>(tile_rows<D>(job, g, a, part0, st, min(a.T, min(tok_end, st + a.ST) - st)), l, pf);
  tile_stage_profile(T, job.profile, H);
  if (TR) tile_signs<D>(smask, job.signs, H);
  __syncthreads();
  tile_positions(T, H);
  tile_groups(T, H, a.tabs);
  const int tab1 = (a.tabs & 1) ? H * (D + 4) : 0;  // V's table behind K's
  if ((a.tabs & 1) && part0 == 0) tile_consts<D, true>(kc, T, g, job.kmeta, 0);
  if ((a.tabs & 2) && part1 == 2) tile_consts<D, true>(kc + tab1, T, g, job.vmeta, 1);
  __syncthreads();
  if (st >= tok_end) return;

  const int h = r % H, tt = r / H;
  const bool native = g.flags & KVMI_F_NATIVE_LAYOUT;
  const int jk = T.pos[0][h], jv = T.pos[1][h];
  const float lvk = (float)T.prof[0][1][jk], lvv = (float)T.prof[1][1][jv];
  const uint2 gk = T.group[0][h], gv = T.group[1][h];
  uint4 hp[2], hn[2];
  if (TR) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      hp[kt] = hadamard_tile_d(kt, false);
      hn[kt] = hadamard_tile_d(kt, true);
    }
  }
  uint32_t over = 0;

  for (; st < tok_end; st += step) {
    const int ste = min(tok_end, st + a.ST);
#pragma unroll 1  // one copy of the section's code for both parts
    for (int part = part0; part < part1; ++part) {
      const bool table = (a.tabs >> part) & 1;
      const int jpos = part ? jv : jk;
      const float lev = part ? lvv : lvk;
      for (int ta = st; ta < ste; ta += a.T) {
        const int nt = min(a.T, ste - ta);
#pragma unroll
        for (int u = 0; u < KS; ++u) pin(pf[u]);
        // rearrange through the wave's buffer: the MFMA operands of the row (piece 2 s + hl of
        // step s), or without a transform its values in output order
        uint4 x[2 * NC];
#pragma unroll
        for (int gi = 0; gi < TG::NG; ++gi) {
#pragma unroll
          for (int v = 0; v < TG::KG; ++v) tb[tile_slot_of<D>(v, l)] = pf[gi * TG::KG + v];
          const uint4* row = tb + r * PP;
          if constexpr (TR) {
#pragma unroll
            for (int s = 0; s < TG::KG; ++s) x[gi * TG::KG + s] = row[2 * s + hl];
          } else {
#pragma unroll
            for (int c = 0; c < (TG::KG + 1) / 2; ++c) {
              const int at = 4 * c + (TG::kTail && c == NC - 1 ? 0 : 2 * hl);
              x[gi * TG::KG + 2 * c] = row[at];
              x[gi * TG::KG + 2 * c + 1] = row[at + 1];
            }
          }
        }
        // the next tile of this wave (unconditional: at the end this tile again, a cache hit)
        int np = part, nta = ta + a.T;
        if (nta >= ste) {
          const bool last = part + 1 == part1;
          np = last ? part0 : part + 1;
          nta = last ? st + step : st;
          if (nta >= tok_end) np = part, nta = ta;
        }
        const int nse = min(tok_end, (nta >= st + step ? st + step : st) + a.ST);
        tile_load<D>(tile_rows<D>(job, g, a, np, nta, min(a.T, nse - nta)), l, pf);

        const bool live = tt < nt;
        if constexpr (TR) {
          const uint4* sm = reinterpret_cast<const uint4*>(smask + opaque(h * (D / 2 + 4))) + hl;
#pragma unroll
          for (int s = 0; s < KS; ++s) x[s] = xor4(x[s], sm[2 * s]);
        }
        // the 16 values of output tile cp as bf16 pairs
        auto values = [&](auto cpc, uint32_t (&y)[8]) {
          constexpr int cp = decltype(cpc)::value;
          if constexpr (TR) {
            constexpr float sc = kTileScale<D, cp>;
            const f32x16 acc = tile_transform<D, cp>(x, hp, hn, [](uint4 A, uint4 B, f32x16 c) { return mfma(A, B, c); });
#pragma unroll
            for (int i = 0; i < 8; ++i) y[i] = pack_bf16x2(acc[2 * i] * sc, acc[2 * i + 1] * sc);
          } else {
            const uint4 u0 = x[2 * cp], u1 = x[2 * cp + 1];
            y[0] = u0.x, y[1] = u0.y, y[2] = u0.z, y[3] = u0.w;
            y[4] = u1.x, y[5] = u1.y, y[6] = u1.z, y[7] = u1.w;
          }
        };
        // bytes of this row in the image
        uint8_t* out = img + (native ? ((ta - st + tt) * H + jpos) * RB : jpos * a.pitch + (ta - st + tt) * RB);
        uint32_t ov = 0;
        if (table) {
          const float2* kq = kc + opaque((part ? tab1 : 0) + h * (D + 4) + 16 * hl);
          tile_each<NC>([&](auto cpc) {
            constexpr int cp = decltype(cpc)::value;
            uint32_t y[8];
            values(cpc, y);
            const int tail = TG::kTail && cp == NC - 1 ? -16 * hl : 0;
            float q[16];
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
              const float4 c = *reinterpret_cast<const float4*>(kq + tail + 32 * cp + i);
              float t0, t1;
              tile_diff(y[i / 2], c.x, c.z, t0, t1);
              q[i] = clamp_level(rbf(t0 * c.y), lev);
              q[i + 1] = clamp_level(rbf(t1 * c.w), lev);
            }
            pack16_bits<BITS>(bits, q, out + (2 * cp + hl) * 2 * bits, live && tile_half_ok<D, cp>(hl), ov);
            chunk_fence();
          });
        } else {
          uint32_t y[NC][8];
          float mn = __builtin_inff(), mx = -__builtin_inff();
          tile_each<NC>([&](auto cpc) {
            constexpr int cp = decltype(cpc)::value;
            values(cpc, y[cp]);
#pragma unroll
            for (int i = 0; i < 8; i += 2) {
              const float e0 = bf_lo(y[cp][i]), e1 = bf_hi(y[cp][i]), e2 = bf_lo(y[cp][i + 1]), e3 = bf_hi(y[cp][i + 1]);
              mn = fminf(fminf(mn, e0), fminf(e1, fminf(e2, e3)));
              mx = fmaxf(fmaxf(mx, e0), fmaxf(e1, fmaxf(e2, e3)));
            }
            chunk_fence();
          });
          const uint2 grp = part ? gv : gk;
          tile_group_minmax(grp, r - h, H, mn, mx);
          const float sc = quant_scale(mn, mx, (int)lev), nrcp = -1.0f / sc;
          if (live && hl == 0 && (grp.y >> 16)) {
            uint16_t* meta = part ? job.vmeta : job.kmeta;
            const int gi = (int)((grp.y >> 8) & 0xffu);
            gst(meta + (int64_t)gi * ntok + ta + tt, (uint16_t)f32_to_bf16_bits(mn));
            gst(meta + (int64_t)(g.G + gi) * ntok + ta + tt, (uint16_t)f32_to_bf16_bits(sc));
          }
          tile_each<NC>([&](auto cpc) {
            constexpr int cp = decltype(cpc)::value;
            float q[16];
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
              float t0, t1;
              tile_diff(y[cp][i / 2], mn, mn, t0, t1);
              q[i] = clamp_level(rbf(t0 * nrcp), lev);
              q[i + 1] = clamp_level(rbf(t1 * nrcp), lev);
            }
            pack16_bits<BITS>(bits, q, out + (2 * cp + hl) * 2 * bits, live && tile_half_ok<D, cp>(hl), ov);
            chunk_fence();
          });
        }
        over |= live ? ov : 0u;
      }
      const int n = ste - st;
      flush_image(img, a.pitch, a.runs, n * RB * (native ? H : 1), tile_stream(job, g, part, 0, st, ntok, RB),
                  (uint32_t)ntok * (uint32_t)RB, l);
    }
  }
  const uint32_t width = 0x01010101u * (0xffu & ~((1u << bits) - 1u));
  if (over & width) atomicOr(err, KVMI_ERR_SYMBOL_RANGE);
}

template <int D, bool TR, int BITS>
int launch_b(const Geo& g, const kvmi_layer_job* jobs, int32_t nj, int32_t mb, int32_t* err, hipStream_t st) {
  const TileArgs a = tile_plan(g, mb, nj, tile_occ(D));
  const unsigned gx = (unsigned)(((int64_t)mb * g.S + a.run - 1) / a.run);
  const size_t lds = (size_t)a.off_wave + (size_t)kTileWaves * a.wave_bytes;
  hipLaunchKernelGGL((tile_encode_kernel<D, TR, BITS>), dim3(gx, (unsigned)nj, a.parts == 1 ? 2 : 1), dim3(kTileThreads),
                     lds, st, g, a, jobs, err);
  return hipGetLastError() == hipSuccess ? KVMI_OK : KVMI_ELAUNCH;
}
template <int D, bool TR>
int launch_d(const Geo& g, const kvmi_layer_job* jobs, int32_t nj, int32_t mb, int32_t* err, hipStream_t st) {
  return g.bits == 4 ? launch_b<D, TR, 4>(g, jobs, nj, mb, err, st) : launch_b<D, TR, 0>(g, jobs, nj, mb, err, st);
}

}  // namespace

int tile_encode(const Geo& g, const kvmi_layer_job* jobs, int32_t nj, int32_t mb, int32_t* err, hipStream_t st) {
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
