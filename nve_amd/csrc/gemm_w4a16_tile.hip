// gemm_w4a16_tile.hip -- W4A16 prefill GEMM for gfx950: Y[M, N] = X[M, K] W[N, K]^T
// with int4 weights in the reference GPU layout and fp16 / bf16 activations, fp32
// accumulation.  Same product as the reference's prefill path (GpuWeight::matmul_x,
// src/gpu_layer.rs:219-237: nve_dequant_w4a16, cuda/nve_kernels.cu:397-433, then a dense
// GEMM), with every weight dequantized exactly as that dequant rounds it
// (f32 fma(n, s, -8 s) = (n - 8) s [times awq[k] in f32], then RNE to the activation type)
// but only in registers.
//
// Work split: a workgroup of 8 waves (two per SIMD, so that one wave's dequantization and LDS
// reads run beside the other's MFMAs) computes a BM x BN tile.  Every wave owns BM x 64
// outputs (TI x 2 tiles of v_mfma_f32_32x32x16) and an equal share of K: WN waves side by side
// cover BN, their KG = 8 / WN groups each take one Q4 block (32 of K) of every iteration, and
// the groups' sums meet in LDS at the end.  So a weight is dequantized once per workgroup and
// each activation read from LDS feeds two MFMAs; sharing K between the waves instead of
// columns is what allows both at these tile sizes.
//   * Global -> LDS transfers only (buffer_load ... lds), in whole 64-byte pieces of a weight
//     row: nibbles for 128 of K per slot, scales (and AWQ factors) for 512 of K (4-byte scale
//     transfers per iteration cost as much as the nibbles').  Activations run 3 iterations
//     ahead (2 with 128 x 128 tiles), nibbles 3-4.
//   * One barrier per iteration, behind which the MFMAs start at once: their k-step 0 operands
//     were read and dequantized in the iteration before.
//   * The transfers and the dequantization are spread over scheduling regions of two MFMAs.
// What bounds it: the VALU and the MFMAs of an iteration are nearly equal (a wave: 16 MFMAs of
// 32.5 cycles; 32 weights per lane of about 18 cycles, the conversions v_cvt_f32_ubyte and
// v_cvt_pk taking 7.5 each) and a full chip clocks lower (0.77 us per 128 x 128 x 128
// iteration with 32-128 workgroups, 1.04 with 256).  Knockouts, 8B gate M = 512, 128 x 256 tiles,
// 77 us: no transfers 60, no dequantization 61, neither 51, no MFMAs 48.
// 8B gate, fp16, us, M = 128 / 256 / 512: 26.9 / 37.6 / 68.9, and q_proj 16.8 / 21.8 / 28.4; a
// kernel of 4 waves (one per SIMD) with 64 of K per slice, which this one replaced: 32.3 /
// 46.0 / 73.8 and 22.7 / 24.3 / 34.6.
#include "common.h"
#include "lds_ring.h"
#include "gemm_tile_plan.h"
#include "w4_launch.h"

namespace nve {

constexpr int kTlWaves = 8;

typedef _Float16 tl_h8_t __attribute__((ext_vector_type(8)));
typedef __bf16 tl_b8_t __attribute__((ext_vector_type(8)));
typedef float tl_f16x_t __attribute__((ext_vector_type(16)));
typedef float tl_f4_t __attribute__((ext_vector_type(4)));
typedef float tl_f2_t __attribute__((ext_vector_type(2)));
typedef _Float16 tl_h2_t __attribute__((ext_vector_type(2)));
typedef __bf16 tl_b2_t __attribute__((ext_vector_type(2)));

// One workgroup: a BM x BN tile by 8 waves, WN of them side by side (64 columns each) in KG =
// 8 / WN groups that split K.  LDS: 4 activation slots (BM rows x KG blocks of 64 B), 3 nibble
// slots (BN rows x 4 blocks of 16 B), 2 scale slots (BN rows x 16 blocks), with AWQ the
// factors of the same 16 blocks; the final exchange of the K groups' sums reuses it.
template <int TI, int WN, bool AWQ>
struct TileCfg {
  static constexpr int KG = kTlWaves / WN;
  static constexpr int BM = 32 * TI, BN = 64 * WN;
  static constexpr int IK = 32 * KG;           // K of one iteration
  static constexpr int NIT = 128 / IK;         // iterations per nibble slot
  static constexpr int SIT = 512 / IK;         // iterations per scale slot
  static constexpr int X = BM * 64 * KG, NIB = BN * 64, SC = BN * 64, AW = AWQ ? 2048 : 0;
  // 128 x 128 tiles leave room for 3 activation slots (one iteration ahead less)
  static constexpr int XS = TI == 4 && WN == 2 ? 3 : 4;
  static constexpr int N0 = XS * X, S0 = N0 + 3 * NIB, A0 = S0 + 2 * SC;
  static constexpr int RING = A0 + 2 * AW;
  static constexpr int RED = kTlWaves * TI * 16 * 256;  // half of every wave's sums
  static constexpr int BYTES = RING > RED ? RING : RED;
  static_assert(BYTES <= 160 * 1024, "LDS");
};

template <bool BF16>
__device__ __forceinline__ tl_f16x_t tl_mfma(u32x4_t a, u32x4_t b, tl_f16x_t c) {
  if (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(tl_b8_t, a), __builtin_bit_cast(tl_b8_t, b), c,
                                                   0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(tl_h8_t, a), __builtin_bit_cast(tl_h8_t, b), c, 0,
                                                0, 0);
}

template <bool BF16>
__device__ __forceinline__ uint32_t tl_pack2(float a, float b) {
  // each value is an f32 first (the fma's rounding), then one v_cvt_pk_{f16,bf16}_f32
  // (round to nearest even): the reference dequant's two roundings
  asm("" : "+v"(a), "+v"(b));
  if (BF16) return __builtin_bit_cast(uint32_t, __builtin_convertvector((tl_f2_t){a, b}, tl_b2_t));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((tl_f2_t){a, b}, tl_h2_t));
}
// The reference dequant of 4 nibbles, one per byte of d (already masked) [times the AWQ
// factors a, each an f32 product of the f32 dequantized value as the reference forms it,]
// rounded to the activation type and packed in k order.
template <bool BF16, bool AWQ>
__device__ __forceinline__ u32x2_t tl_dequant4(uint32_t d, float s, float s8, const tl_f4_t& a) {
  // the masked dword is opaque to the compiler, so each byte goes through one
  // v_cvt_f32_ubyte{0..3} (instead of a bit-field extract and a conversion)
  asm("" : "+v"(d));
  float v[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    v[t] = fmaf((float)((d >> (8 * t)) & 0xffu), s, s8);
    if constexpr (AWQ) v[t] *= a[t];
  }
  u32x2_t r;
  r.x = tl_pack2<BF16>(v[0], v[1]);
  r.y = tl_pack2<BF16>(v[2], v[3]);
  return r;
}

typedef __attribute__((address_space(3))) char tl_lds_t;

// What a wave holds of one iteration's weights: per column tile the 8 nibble bytes of its
// k-run and the block scale, and with AWQ the 8 factors of each of the two k-steps.
template <bool AWQ>
struct TileRaw {
  u32x2_t q[2];
  float s[2];
  tl_f4_t aw[AWQ ? 4 : 1];
};

// Quarter c of a k-step's two B operands: values 4 (c % 2) .. + 3 of column tile c / 2.
template <bool BF16, bool AWQ, int KK>
__device__ __forceinline__ void tl_b_quarter(u32x4_t (&f)[2], const TileRaw<AWQ>& w, int c) {
  const int j = c >> 1;
  const uint32_t q = (c & 1) ? w.q[j].y : w.q[j].x;
  const u32x2_t v = tl_dequant4<BF16, AWQ>(KK ? (q >> 4) & 0x0F0F0F0Fu : q & 0x0F0F0F0Fu, w.s[j], -8.0f * w.s[j],
                                           w.aw[AWQ ? 2 * KK + (c & 1) : 0]);
  if (c & 1) {
    f[j].z = v.x;
    f[j].w = v.y;
  } else {
    f[j].x = v.x;
    f[j].y = v.y;
  }
}

// SPLIT: blockIdx.y = z takes iterations z ks .. z ks + ks - 1 of K and stores its fp32
// partial tile to out + z M N (tl_reduce_kernel adds the partials in order).
template <bool BF16, bool AWQ, int OUT_DT, int TI, int WN, bool SPLIT>
__global__ __launch_bounds__(64 * kTlWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_w4a16_tile_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ nib, const float* __restrict__ sc,
    const float* __restrict__ awq, void* __restrict__ out, int M, int N, int K, int n_tiles, int ks) {
  static_assert(!SPLIT || OUT_DT == NVE_DT_F32, "split partials are fp32");
#ifdef __HIP_DEVICE_COMPILE__  // (the host pass has no use for the body and cannot lower its LDS accesses)
  extern __shared__ __align__(16) char tl_smem[];
  using C = TileCfg<TI, WN, AWQ>;
  constexpr int KG = C::KG, BM = C::BM, BN = C::BN;
  static_assert(KG == 2 || KG == 4, "K groups");
  constexpr int XT = 2 * TI * KG;                   // activation transfers (1 KiB) of an iteration
  constexpr int NX = (XT + kTlWaves - 1) / kTlWaves;  // per wave, at most
  constexpr int NXMIN = XT / kTlWaves;                // and at least
  constexpr int NS = BN / 16 / kTlWaves;              // scale transfers per wave and slot
  constexpr int RS = 64 * KG, NCH = 4 * KG;  // LDS row bytes / 16-byte chunks of an activation row
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = wave / WN, wn = wave % WN;

  // XCD-grouped tile order: block b runs on XCD b % 8; the blocks of one XCD take
  // consecutive linear tiles (row block major)
  const int total = gridDim.x, b = blockIdx.x, xcd = b & 7;
  const int per = total >> 3, extra = total & 7;
  const int lin = xcd * per + min(xcd, extra) + (b >> 3);
  const int m0 = (lin / n_tiles) * BM, n0 = (lin % n_tiles) * BN;
  // this workgroup's iterations: t0 .. t0 + T - 1 (t0 a multiple of the nibble slot's)
  const int t0 = SPLIT ? (int)blockIdx.y * ks : 0;
  const int T = SPLIT ? min(K / C::IK - t0, ks) : K / C::IK;

  // buffer resources (raw buffers, 32-bit offsets: the host routes larger operands elsewhere;
  // a read past the end of the scales or factors -- the last slot of a K that is no multiple
  // of 512 -- returns 0): per-lane offset in a VGPR, the iteration's in an SGPR
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)x, (short)0, 2 * M * K, 0x00020000);
  const __amdgpu_buffer_rsrc_t nr = __builtin_amdgcn_make_buffer_rsrc((void*)nib, (short)0, N * (K / 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc((void*)sc, (short)0, N * (K / 8), 0x00020000);
  const __amdgpu_buffer_rsrc_t ar =
      __builtin_amdgcn_make_buffer_rsrc((void*)(AWQ ? awq : sc), (short)0, AWQ ? 4 * K : 0, 0x00020000);
  // activation transfers: instruction i fills 1024 / RS tile rows; lane l writes row l / NCH of
  // them at chunk position l % NCH, i.e. global chunk position ^ swizzle(row)
  auto swz = [](int r) { return KG == 4 ? (r & 15) : ((r >> 1) & 7); };
  uint32_t xoff[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int r = (kTlWaves * i + wave) * (1024 / RS) + lane / NCH;
    const int c = (lane % NCH) ^ swz(r);
    xoff[i] = ((uint32_t)min(m0 + r, M - 1) * (uint32_t)K + 8u * c) * 2u;
  }
  // weight transfers (1 KiB: 16 rows x 64 B): lane l carries row 16 i + l / 4 of the tile, 16-byte
  // position l % 4, which holds chunk (position - row / 4) % 4 of the slot's 64 bytes (so that the
  // rows read together fall on different banks)
  constexpr int NW = BN / 16 / kTlWaves;  // row groups per wave
  uint32_t noff[NW], soff[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int r = 16 * (kTlWaves * i + wave) + (lane >> 2);
    const uint32_t rg = (uint32_t)min(n0 + r, N - 1), c = ((lane & 3) - (r >> 2)) & 3;
    noff[i] = rg * (uint32_t)(K / 2) + 16u * c;
    soff[i] = rg * (uint32_t)(K / 8) + 16u * c;
  }

  // A fragments: rows 32 i + l % 32, chunk 4 g + 2 kk + l / 32 of the row
  const int fr = lane & 31, fhi = lane >> 5;
  const uint32_t a0 = fr * RS + 16 * ((4 * g + fhi) ^ swz(fr)), a1 = fr * RS + 16 * ((4 * g + 2 + fhi) ^ swz(fr));
  // B operands: column tile j of the wave covers rows 64 wn + 32 j + l % 32; nibble bytes
  // 8 (l / 32) .. + 7 of the group's block: low nibbles are k-step 0's values, high ones k-step 1's
  const int wrow = 64 * wn + fr, wq = wrow >> 2;
  const uint32_t bq = wrow * 64 + 16 * ((g + wq) & 3) + 8 * fhi;
  constexpr int TSTEP = 32 * 64;  // column tile 1

  tl_f16x_t acc[2 * TI];  // [2 i + j]
#pragma unroll
  for (int i = 0; i < 2 * TI; ++i) acc[i] = tl_f16x_t{};

  tl_lds_t* const lds = (tl_lds_t*)tl_smem;
  // transfers (iterations and slots past the end re-read the last ones, which keeps every
  // iteration's transfer count equal)
  auto issue_x = [&](int e, tl_lds_t* d, int t) __attribute__((always_inline)) {
    if (XT % kTlWaves == 0 || kTlWaves * e + wave < XT)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void_t*)(d + (kTlWaves * e + wave) * 1024), 16, xoff[e],
                                               (t0 + min(t, T - 1)) * (64 * KG), 0, 0);
  };
  const int pmax = (T - 1) / C::NIT, p0 = t0 / C::NIT;
  auto issue_nib = [&](int i, tl_lds_t* d, int p) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(nr, (lds_void_t*)(d + (kTlWaves * i + wave) * 1024), 16, noff[i],
                                             (p0 + min(p, pmax)) * 64, 0, 0);
  };
  const int smax = (T - 1) / C::SIT;
  auto issue_sc = [&](tl_lds_t* d, tl_lds_t* da, int p) __attribute__((always_inline)) {
    const int pc = min(p, smax);
#pragma unroll
    for (int i = 0; i < NS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(sr, (lds_void_t*)(d + (kTlWaves * i + wave) * 1024), 16, soff[i],
                                               t0 * (4 * KG) + pc * 64, 0, 0);
    if (AWQ && wave < 2)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ar, (lds_void_t*)(da + wave * 1024), 16, wave * 1024 + lane * 16,
                                               t0 * (128 * KG) + pc * 2048, 0, 0);
  };
  // the raw weights of iteration u (its nibble slot nb, scale slot sb, factors ab)
  auto read_raw = [&](TileRaw<AWQ>& w, const tl_lds_t* nb, const tl_lds_t* sb, const tl_lds_t* ab, int u)
      __attribute__((always_inline)) {
    const uint32_t q = C::NIT == 2 ? bq ^ ((u & 1) << 5) : bq;  // block 2 (u % 2) + g of the slot
    const int blk = (u % C::SIT) * KG + g;                      // of the scale slot's 16
    const uint32_t s = wrow * 64 + 16 * (((blk >> 2) + wq) & 3) + 4 * (blk & 3);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      w.q[j] = *(const __attribute__((address_space(3))) u32x2_t*)(nb + q + j * TSTEP);
      w.s[j] = *(const __attribute__((address_space(3))) float*)(sb + s + j * TSTEP);
    }
    if constexpr (AWQ) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        w.aw[i] = *(const __attribute__((address_space(3))) tl_f4_t*)(ab + blk * 128 + 32 * fhi + (i & 1) * 16 +
                                                                      (i >> 1) * 64);
    }
  };
  auto read_a = [&](u32x4_t (&f)[TI], const tl_lds_t* xs, uint32_t a) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TI; ++i) f[i] = *(const __attribute__((address_space(3))) u32x4_t*)(xs + a + i * 32 * RS);
  };

  // Pipeline: iteration u issues the activations of u + 3, its share of a nibble slot 3 (KG = 4)
  // or 2 (KG = 2: two iterations each) ahead and, as the first of a scale slot, the next one;
  // it reads the k-step 0 activations and the raw weights of u + 1 and forms that step's
  // operands, so that the next iteration's MFMAs start right behind its barrier.
  constexpr int PD = C::NIT == 2 ? 2 : 3;  // nibble slots ahead
  issue_sc(lds + C::S0, lds + C::A0, 0);
#pragma unroll
  for (int p = 0; p < PD; ++p)
#pragma unroll
    for (int i = 0; i < NW; ++i) issue_nib(i, lds + C::N0 + p * C::NIB, p);
#pragma unroll
  for (int i = 0; i < C::XS - 1; ++i)
#pragma unroll
    for (int e = 0; e < NX; ++e) issue_x(e, lds + i * C::X, i);
  u32x4_t fa[TI], fb[2];
  TileRaw<AWQ> cur;
  wait_vmcnt<C::XS == 4 ? NXMIN : 0>();
  lds_barrier();
  // (the slots read and those the transfers fill are different objects to the compiler
  // (restrict), so it adds no waits of its own for the transfers)
  auto first = [&](const tl_lds_t* __restrict__ r, tl_lds_t* __restrict__ none) __attribute__((always_inline)) {
    read_a(fa, r, a0);
    read_raw(cur, r + C::N0, r + C::S0, r + C::A0, 0);
  };
  first(lds, lds + C::X);
#pragma unroll
  for (int c = 0; c < 4; ++c) tl_b_quarter<BF16, AWQ, 0>(fb, cur, c);

  auto iter = [&](const tl_lds_t* __restrict__ rd, tl_lds_t* __restrict__ wr, int x0, int x1, int n1, int s1, int xd,
                  int nd, int sd, int u) __attribute__((always_inline)) {
    u32x4_t fa1[TI], fb1[2];
    TileRaw<AWQ> nxt;
    read_a(fa1, rd + x0 * C::X, a1);
    read_raw(nxt, rd + C::N0 + n1 * C::NIB, rd + C::S0 + s1 * C::SC, rd + C::A0 + s1 * C::AW, u + 1);
    // one scheduling region per two MFMAs, each with its share of the transfers and of the
    // next k-step's dequantization: left in one group the transfers of the eight waves
    // hold the address pipeline while no MFMA runs
    auto extra = [&](int r) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < NX; ++e)
        if (r == e) issue_x(e, wr + xd * C::X, u + C::XS - 1);
      if (r == TI) {
        if constexpr (C::NIT == 1) {
          issue_nib(0, wr + C::N0 + nd * C::NIB, u + 3);
        } else if ((u & 1) == 0) {
          issue_nib(0, wr + C::N0 + nd * C::NIB, (u >> 1) + 2);
        } else {
          issue_nib(NW - 1, wr + C::N0 + nd * C::NIB, (u >> 1) + 2);
        }
      }
      if (r == TI + 1 && u % C::SIT == 0) issue_sc(wr + C::S0 + sd * C::SC, wr + C::A0 + sd * C::AW, u / C::SIT + 1);
    };
#pragma unroll
    for (int i = 0; i < TI; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[2 * i + j] = tl_mfma<BF16>(fa[i], fb[j], acc[2 * i + j]);
      extra(i);
#pragma unroll
      for (int c = 4 * i / TI; c < 4 * (i + 1) / TI; ++c) tl_b_quarter<BF16, AWQ, 1>(fb1, cur, c);
      __builtin_amdgcn_sched_barrier(0);
    }
    read_a(fa, rd + x1 * C::X, a0);
#pragma unroll
    for (int i = 0; i < TI; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[2 * i + j] = tl_mfma<BF16>(fa1[i], fb1[j], acc[2 * i + j]);
      extra(TI + i);
#pragma unroll
      for (int c = 4 * i / TI; c < 4 * (i + 1) / TI; ++c) tl_b_quarter<BF16, AWQ, 0>(fb, nxt, c);
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = nxt;
  };
  static_assert(NX <= TI, "one activation transfer per region");
  int xs = 0, ns = 0;  // slots of iteration u's activations and nibbles
  for (int u = 0; u < T; ++u) {
    // all but the transfers of iteration u - 1 have landed (3 activation slots: its
    // activations, the first it issued, too)
    wait_vmcnt<C::XS == 4 ? NXMIN + 1 : 1>();
    lds_barrier();
    const int nn = C::NIT == 1 || (u & 1) ? (ns == 2 ? 0 : ns + 1) : ns;  // of iteration u + 1
    const int nd = C::NIT == 1 ? ns : (ns == 0 ? 2 : ns - 1);              // (u + 3) % 3 / (u / 2 + 2) % 3
    const int s1 = ((u + 1) / C::SIT) & 1, sd = (u / C::SIT + 1) & 1;
    const int x1 = xs == C::XS - 1 ? 0 : xs + 1;
    iter(lds, lds, xs, x1, nn, s1, xs == 0 ? C::XS - 1 : xs - 1, nd, sd, u);
    xs = x1;
    ns = nn;
  }
  // the transfers issued past the last iteration land before the LDS is reused or released
  wait_vmcnt<0>();
  lds_barrier();

  // sums of the K groups: group g and g ^ (KG / 2) exchange halves of their tiles, then (KG =
  // 4) g and g ^ 1 halves of what is left; every group ends with 2 TI / KG tiles of the sum
  // (each exchange is one fp32 addition of the same two values in either order: the same
  // bits whichever wave adds them)
  constexpr int LEFT = 2 * TI / KG;
  static_assert(LEFT >= 1, "tiles per group");
  auto put = [&](int cnt, int from) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < cnt; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const tl_f16x_t& v = acc[from + t];
        *(__attribute__((address_space(3))) tl_f4_t*)(lds + ((wave * cnt + t) * 4 + r) * 1024 + lane * 16) =
            (tl_f4_t){v[4 * r], v[4 * r + 1], v[4 * r + 2], v[4 * r + 3]};
      }
  };
  auto add = [&](int cnt, int from, int partner) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < cnt; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const tl_f4_t v =
            *(const __attribute__((address_space(3))) tl_f4_t*)(lds + ((partner * cnt + t) * 4 + r) * 1024 + lane * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][4 * r + e] = acc[from + t][4 * r + e] + v[e];
      }
  };
  int f0 = 0;  // first tile this group holds
  if (g < KG / 2) {
    put(TI, TI);
    lds_barrier();
    add(TI, 0, wave ^ 4);
  } else {
    put(TI, 0);
    lds_barrier();
    add(TI, TI, wave ^ 4);
    f0 = TI;
  }
  if constexpr (KG == 4) {
    lds_barrier();
    if (!(g & 1)) {
      put(TI / 2, TI / 2);
      lds_barrier();
      add(TI / 2, 0, wave ^ WN);
    } else {
      put(TI / 2, 0);
      lds_barrier();
      add(TI / 2, TI / 2, wave ^ WN);
      f0 += TI / 2;
    }
  }

  // 32 x 32 result layout: register r of lane l holds D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32]
  const size_t z0 = SPLIT ? (size_t)blockIdx.y * M * N : 0;
  auto store = [&](bool check) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < LEFT; ++t) {
      const int f = f0 + t;
      const int n = n0 + 64 * wn + 32 * (f & 1) + fr, mt = m0 + 32 * (f >> 1) + 4 * fhi;
      const size_t o = z0 + (size_t)mt * N + n;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dm = 8 * (r >> 2) + (r & 3);
        if (check && !(mt + dm < M && n < N)) continue;
        store_out<OUT_DT>(out, o + (size_t)dm * N, acc[t][r]);
      }
    }
  };
  if (m0 + BM <= M && n0 + BN <= N)
    store(false);
  else
    store(true);
#endif
}

// out[i] = sum over z = 0 .. split - 1 of part[z n + i], in that order, rounded to OUT_DT.
// V consecutive elements per thread (V = 4 where n is a multiple of 4: 16-byte loads).
template <int OUT_DT, int V>
__global__ __launch_bounds__(256) void tl_reduce_kernel(const float* __restrict__ part, void* __restrict__ out,
                                                        size_t n, int split) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * V;
  if (i >= n) return;
  typedef float fv_t __attribute__((ext_vector_type(V)));
  fv_t y = *(const fv_t*)(part + i);
#pragma unroll 4
  for (int z = 1; z < split; ++z) y += *(const fv_t*)(part + (size_t)z * n + i);
#pragma unroll
  for (int e = 0; e < V; ++e) store_out<OUT_DT>(out, i + e, y[e]);
}

}  // namespace nve

namespace nve_host {

// The tile kernel serves K % 128 == 0, where every byte offset fits its buffer resource
// (activations 2 M K, nibbles N K / 2, scales N K / 8, factors 4 K bytes below 2^31), with
// 16-byte aligned scales (its transfers take 4 scales at a time).
bool gemm_tile_fits(int M, int N, int K, const void* sc) {
  return K % 128 == 0 && M >= 1 && N >= 1 && (long)M * K < (1L << 30) && (long)N * (K / 2) < (1L << 31) &&
         aligned(sc, 16);
}

// fp32 partial bytes a caller's workspace is sized for: a 128 x 128 tile grid split over K
// while it stays within one workgroup per CU and 512 of K per split.
size_t gemm_tile_parts_bytes(int M, int N, int K) {
  if (!gemm_tile_fits(M, N, K, nullptr)) return 0;
  const long g = (long)((M + 127) / 128) * ((N + 127) / 128);
  const int kit = K / 128;
  const int by_grid = g >= 256 ? 1 : (int)(256 / g), by_k = kit / 4 > 1 ? kit / 4 : 1;
  const int split = by_grid < by_k ? by_grid : by_k;
  const int per = (kit + split - 1) / split, used = (kit + per - 1) / per;
  return used > 1 ? (size_t)used * M * N * sizeof(float) : 0;
}

template <bool BF16, bool AWQ, int OUT_DT, int TI, int WN, bool SPLIT>
static hipError_t launch_tile_k(const void* x, int M, const uint8_t* nib, const float* sc, const float* awq, void* out,
                                int N, int K, int split, int ks, hipStream_t s) {
  using C = nve::TileCfg<TI, WN, AWQ>;
  auto kern = nve::gemm_w4a16_tile_kernel<BF16, AWQ, OUT_DT, TI, WN, SPLIT>;
  static thread_local int attr_dev = -1;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (attr_dev != dev) {
    e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::BYTES);
    if (e != hipSuccess) return e;
    attr_dev = dev;
  }
  const int nt = (N + C::BN - 1) / C::BN, mt = (M + C::BM - 1) / C::BM;
  hipLaunchKernelGGL(kern, dim3(nt * mt, split), dim3(64 * nve::kTlWaves), C::BYTES, s, (const uint16_t*)x, nib, sc,
                     awq, out, M, N, K, nt, ks);
  return hipGetLastError();
}

template <bool BF16, bool AWQ, int OUT_DT, bool SPLIT>
static hipError_t launch_tile_t(const TilePlan& p, const void* x, int M, const uint8_t* nib, const float* sc,
                                const float* awq, void* out, int N, int K, hipStream_t s) {
  switch (p.shape) {
    case 0: return launch_tile_k<BF16, AWQ, OUT_DT, 2, 2, SPLIT>(x, M, nib, sc, awq, out, N, K, p.split, p.ks, s);
    case 1: return launch_tile_k<BF16, AWQ, OUT_DT, 4, 2, SPLIT>(x, M, nib, sc, awq, out, N, K, p.split, p.ks, s);
    case 2: return launch_tile_k<BF16, AWQ, OUT_DT, 3, 4, SPLIT>(x, M, nib, sc, awq, out, N, K, p.split, p.ks, s);
    default: return launch_tile_k<BF16, AWQ, OUT_DT, 4, 4, SPLIT>(x, M, nib, sc, awq, out, N, K, p.split, p.ks, s);
  }
}

template <int OUT_DT>
static void launch_reduce(const float* parts, void* out, size_t n, int split, hipStream_t s) {
  if (n % 4 == 0 && aligned(out, OUT_DT == NVE_DT_F32 ? 16 : 8))
    hipLaunchKernelGGL((nve::tl_reduce_kernel<OUT_DT, 4>), dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s,
                       parts, out, n, split);
  else
    hipLaunchKernelGGL((nve::tl_reduce_kernel<OUT_DT, 1>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, parts,
                       out, n, split);
}

template <bool BF16, bool AWQ>
static hipError_t launch_tile_x(const TilePlan& p, const void* x, int M, const uint8_t* nib, const float* sc,
                                const float* awq, void* out, int out_dt, int N, int K, float* parts, hipStream_t s) {
  if (p.split > 1) {
    const hipError_t e = launch_tile_t<BF16, AWQ, NVE_DT_F32, true>(p, x, M, nib, sc, awq, parts, N, K, s);
    if (e != hipSuccess) return e;
    const size_t n = (size_t)M * N;
    switch (out_dt) {
      case NVE_DT_F16: launch_reduce<NVE_DT_F16>(parts, out, n, p.split, s); break;
      case NVE_DT_BF16: launch_reduce<NVE_DT_BF16>(parts, out, n, p.split, s); break;
      default: launch_reduce<NVE_DT_F32>(parts, out, n, p.split, s); break;
    }
    return hipGetLastError();
  }
  switch (out_dt) {
    case NVE_DT_F16: return launch_tile_t<BF16, AWQ, NVE_DT_F16, false>(p, x, M, nib, sc, awq, out, N, K, s);
    case NVE_DT_BF16: return launch_tile_t<BF16, AWQ, NVE_DT_BF16, false>(p, x, M, nib, sc, awq, out, N, K, s);
    default: return launch_tile_t<BF16, AWQ, NVE_DT_F32, false>(p, x, M, nib, sc, awq, out, N, K, s);
  }
}

hipError_t launch_gemm_w4a16_tile(const TilePlan& p, const void* x, int x_dt, int M, const uint8_t* nib,
                                  const float* sc, const float* awq, void* out, int out_dt, int N, int K,
                                  float* parts, hipStream_t s) {
  const bool bf = x_dt == NVE_DT_BF16;
  if (awq)
    return bf ? launch_tile_x<true, true>(p, x, M, nib, sc, awq, out, out_dt, N, K, parts, s)
              : launch_tile_x<false, true>(p, x, M, nib, sc, awq, out, out_dt, N, K, parts, s);
  return bf ? launch_tile_x<true, false>(p, x, M, nib, sc, awq, out, out_dt, N, K, parts, s)
            : launch_tile_x<false, false>(p, x, M, nib, sc, awq, out, out_dt, N, K, parts, s);
}

}  // namespace nve_host
