// Fused FlatQuant quantize of float32 activations on the float32 matrix cores
// (v_mfma_f32_16x16x4_f32: the full float32 product and sum, twice the rate of
// the VALU's): fq_f32_kernel, M up to 128, N up to 256.
#include <algorithm>
#include <type_traits>

#include "flatquant_common.h"

namespace qo {

namespace {

// A launch's sizes and LDS plan (byte offsets). inv_n = ceil(2^32 / N), for
// row = umulhi(e, inv_n), exact for e < 2^16.
struct FqF32 {
  int M, N, F, mb, nb;   // mb = ceil(M / 16): MBX or one less; nb = ceil(N / 16), also the 16-deep slabs of the first product
  int tpb;               // token slots per workgroup
  uint32_t inv_n;
  int px;                // X row pitch in floats: 16 nb + 4 (16 rows start on 16 bank groups)
  int xslot;             // bytes of one slot's X rows
  int stage_off, cslot;  // staged codes of slot 0; bytes of a slot
  int alias;             // the codes are staged over X's rows
  int lf_off, red_off;   // L's fragments, the scale exchange
  int pack;
};

__device__ inline v4f mfma4(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Codes of one lane's 4 columns as nibbles (PK, code + 8 in bits 4r) or bytes.
// The quotient is y / s correctly rounded: rcp is 1 / s correctly rounded, so one
// Newton step from y * rcp gives it (Markstein), unless s's mantissa is all ones
// or an operand leaves the normal range, which the caller excludes. Quotients
// beyond 16 keep their side. A NaN gives nibble 0 (code -8) or byte 0, as the
// fallback's casts do.
template <bool PK>
__device__ inline uint32_t f32_codes4(const v4f& y, float s, float rcp) {
  uint32_t w = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float q0 = __builtin_amdgcn_fmed3f(y[r] * rcp, -16.0f, 16.0f);
    const float q = fmaf(fmaf(-q0, s, y[r]), rcp, q0);
    // 1.5 * 2^23 + 8 has a unit ulp: the sum rounds half to even and holds code + 8
    const uint32_t c = __builtin_bit_cast(uint32_t, __builtin_amdgcn_fmed3f(q, -8.0f, 7.0f) + 12582920.0f);
    if constexpr (PK) w |= (c & 0xFu) << (4 * r);
    else w |= (y[r] != y[r] ? 0u : (c - 8u) & 0xFFu) << (8 * r);
  }
  return w;
}
// The same by the fallback's own division (scales of 0, infinity and the excluded ones).
__device__ inline uint32_t f32_codes4_div(const v4f& y, float s, bool pack) {
  uint32_t w = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float q = opaque(y[r]) / s;
    w |= pack ? (uint32_t)(fq_code_from_quot<true>(q) + 8) << (4 * r)
              : (uint32_t)(fq_code_from_quot<false>(q) & 0xFF) << (8 * r);
  }
  return w;
}

// ---------------------------------------------------------------------------
// nb waves share a token, one per block p of 16 columns; small widths put tpb
// tokens into a workgroup. X's rows and L's fragments are in LDS, R's in VGPRs.
//
// Every sum runs over k in order, one rounding per product (the MFMA adds its
// four in lane-group order), so the results are those of fq_generic_kernel, and
// of a host BLAS that sums in order, bit for bit. MFMA j of a 16-deep slab takes
// k = 16 kq + 4 j + lg from lane group lg: a row's 16 columns lie transposed (4 x
// 4) in LDS, so that one 16-byte read feeds four MFMAs. The rows of a block enter
// the first product in the same order, which makes accumulator r of lane group
// lg row 16 rb + 4 r + lg of Z: the second product's A operand as it is.
// Staging of X and of the codes, padding and barriers as in fq_tile_kernel
// (flatquant_tile.h).
//
// R (4 VGPRs per 16-deep slab), X, Z and Y (4 per row block) are all held at
// once: MBX x KQX = 6 x 12 and 8 x 12 spill 17 and 93 VGPRs, 2, 4, 6 and 8 x 16
// (128 registers) 17, 87, 148 and 208; every instance spills SGPRs (25 to 83).
// Those are still 2 times (1024 x 8 x 255) to 9 times (1024 x 64 x 254, 128 x 144)
// faster than fq_generic_kernel.
//
// Bound: the float32 MFMA (64 FLOP per clock and SIMD: a token of 112 x 128 takes
// a CU 11 us), at small widths the launch and set-up. Measured (kernel alone,
// before: fq_generic_kernel): 128 x 64 x 64 10.1 -> 7.8 us, 1000 x 64 x 64 32 ->
// 18 us, 1000 x 96 x 96 163 -> 57 us, 1000 x 112 x 128 830 -> 83 us (83 TFLOP/s).
// ---------------------------------------------------------------------------
template <int MBX, int KQX>
__global__ void __launch_bounds__(KQX <= 8 ? 512 : 64 * KQX)
fq_f32_kernel(const float* __restrict__ x, int64_t tokens, int64_t x_ld, const float* __restrict__ left,
              const float* __restrict__ right, FqF32 d, float clip, void* __restrict__ out_codes,
              float* __restrict__ out_scales) {
  extern __shared__ __align__(16) unsigned char smem[];
  unsigned char* const lf = smem + d.lf_off;

  const int tid = threadIdx.x, nt = blockDim.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nb = d.nb;
  const int tau = wave / nb, p = wave % nb;
  const int li = lane & 15, lg = lane >> 4;
  const int nts = 64 * nb;            // threads of a token slot
  const int st = tid - tau * nts;
  const int M = d.M, N = d.N, F = d.F, px = d.px;
  float* const xs = reinterpret_cast<float*>(smem + tau * d.xslot);
  unsigned char* const cs = smem + d.stage_off + tau * d.cslot;
  float* const red = reinterpret_cast<float*>(smem + d.red_off) + tau * 16;
  const int64_t ngroups = (tokens + d.tpb - 1) / d.tpb;

  // Column k of a row is at slot(k): k = 16 kq + 4 j + i at 16 kq + 4 i + j.
  auto slot = [](int k) { return (k & ~15) | ((k & 3) << 2) | ((k >> 2) & 3); };
  // One token into registers, at most MBX 16-byte chunks per thread, and from
  // there into its rows, in the pieces the row length allows.
  const int nch = F >> 2;
  v4f xr[MBX];
  auto load_x = [&](int64_t t) __attribute__((always_inline)) {
    const char* src = reinterpret_cast<const char*>(x + (t < tokens ? t : tokens - 1) * x_ld);
#pragma unroll
    for (int i = 0; i < MBX; ++i) xr[i] = *reinterpret_cast<const v4f*>(src + 16u * (uint32_t)min(st + i * nts, nch - 1));
  };
  auto write_x = [&]() __attribute__((always_inline)) {
    int s = st;
    asm volatile("" : "+v"(s));   // addresses recomputed per token instead of held in VGPRs
#pragma unroll
    for (int i = 0; i < MBX; ++i) {
      if (s + i * nts >= nch) continue;
      const uint32_t e = 4 * (s + i * nts);
      int row = (int)__umulhi(e, d.inv_n), col = (int)e - row * N;
      if ((N & 3) == 0) {
        float* const at = xs + row * px + (col & ~15) + ((col >> 2) & 3);
#pragma unroll
        for (int k = 0; k < 4; ++k) at[4 * k] = xr[i][k];
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          xs[row * px + slot(col)] = xr[i][k];
          if (++col >= N) { col = 0; ++row; }
        }
      }
    }
  };
  auto zero_pads = [&]() __attribute__((always_inline)) {
    for (int r = st; r < M; r += nts)
      for (int c = N; c < 16 * nb; ++c) xs[r * px + slot(c)] = 0.f;
    for (int i = st; i < (16 * d.mb - M) * (px / 4); i += nts) reinterpret_cast<v4f*>(xs + M * px)[i] = v4f{0.f, 0.f, 0.f, 0.f};
  };

  int64_t g = blockIdx.x;   // grid <= ngroups
  // R: rf[kq][j] = R[16kq + 4j + lg][16p + li], L: fragment (b, kb), element j =
  // L[16kb + 4j + lg][16b + li], both 0 in the padding; 64-byte runs of rows.
  v4f rf[KQX];
  {
    const int n = min(16 * p + li, N - 1);
#pragma unroll
    for (int kq = 0; kq < KQX; ++kq)
#pragma unroll
      for (int j = 0; j < 4; ++j) rf[kq][j] = right[min(16 * kq + 4 * j + lg, N - 1) * N + n];
    load_x(g * d.tpb + tau);
#pragma unroll
    for (int kq = 0; kq < KQX; ++kq)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (16 * p + li >= N || 16 * kq + 4 * j + lg >= N) rf[kq][j] = 0.f;
  }
  zero_pads();
  const int nw = nt >> 6;
  for (int f0 = wave; f0 < MBX * MBX; f0 += 4 * nw) {   // 16 loads in flight
    v4f v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int f = min(f0 + u * nw, MBX * MBX - 1), b = f / MBX, kb = f % MBX;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[u][j] = left[min(16 * kb + 4 * j + lg, M - 1) * M + min(16 * b + li, M - 1)];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int f = f0 + u * nw, b = f / MBX, kb = f % MBX;
      if (f >= MBX * MBX) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (16 * kb + 4 * j + lg >= M || 16 * b + li >= M) v[u][j] = 0.f;
      *reinterpret_cast<v4f*>(lf + f * 1024 + 16 * lane) = v[u];
    }
  }
  write_x();
  lds_barrier();
  if (g + gridDim.x < ngroups) load_x((g + gridDim.x) * d.tpb + tau);

  // A operands (rb, kq) at (16 rb) px + 16 kq: row 4 (li % 4) + li / 4 of the block
  const float* const xa = xs + (4 * (li & 3) + (li >> 2)) * px + 4 * lg;
  const int rem = N - (16 * p + 4 * lg);           // this lane's columns inside the row (4 or more: all)
  const int cbytes = d.pack ? F >> 1 : F;
  const bool full = d.mb == MBX;
  while (true) {
    // First product: z[rb][r] = Z[16rb + 4r + lg][16p + li], two row blocks
    // (independent sums) at a time.
    v4f z[MBX];
#pragma unroll
    for (int rb = 0; rb < MBX; rb += 2) {
      v4f c0 = {0.f, 0.f, 0.f, 0.f}, c1 = {0.f, 0.f, 0.f, 0.f};
      const float* const a0 = xa + 16 * rb * px;
      const float* const a1 = a0 + (rb + 1 < MBX - 1 || full ? 16 * px : 0);   // an absent last block repeats the one before
#pragma unroll
      for (int kq = 0; kq < KQX; ++kq) {
        if (kq >= nb) continue;
        const v4f u = *reinterpret_cast<const v4f*>(a0 + 16 * kq), v = *reinterpret_cast<const v4f*>(a1 + 16 * kq);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          c0 = mfma4(u[j], rf[kq][j], c0);
          c1 = mfma4(v[j], rf[kq][j], c1);
        }
      }
      z[rb] = c0;
      z[rb + 1] = c1;
      // padded rows of Z: 0, whatever R holds (and whatever an absent block repeated)
      if (rb == MBX - 2) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int r = 0; r < 4; ++r) z[rb + e][r] = 16 * (rb + e) + 4 * r + lg < M ? z[rb + e][r] : 0.f;
      }
      __builtin_amdgcn_sched_barrier(0);
    }

    // Second product, transposed: y[b] = Y[16b + li][16p + 4lg .. + 3], two row
    // blocks of Y at a time; max |Y| (the padding's are 0, or NaN, which fmaxf drops).
    v4f y[MBX];
    float amax = 0.f;
#pragma unroll
    for (int b = 0; b < MBX; b += 2) {
      v4f c0 = {0.f, 0.f, 0.f, 0.f}, c1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < MBX; ++kb) {
        if (kb == MBX - 1 && !full) continue;
        const v4f u = *reinterpret_cast<const v4f*>(lf + (b * MBX + kb) * 1024 + 16 * lane);
        const v4f v = *reinterpret_cast<const v4f*>(lf + ((b + 1) * MBX + kb) * 1024 + 16 * lane);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          c0 = mfma4(z[kb][r], u[r], c0);
          c1 = mfma4(z[kb][r], v[r], c1);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) amax = fmaxf(fmaxf(amax, fabsf(c0[r])), fabsf(c1[r]));
      y[b] = c0;
      y[b + 1] = c1;
      __builtin_amdgcn_sched_barrier(0);
    }
    // non-negative floats order like their bits; a token of NaNs alone (each wave
    // then reports all ones) takes an infinite scale, as from the empty extremes
    uint32_t top = wave_max_u32(__builtin_bit_cast(uint32_t, amax));
    if (top == 0u) {
      bool any = false;
      int rows = M - li, cols = rem;
      asm volatile("" : "+v"(rows), "+v"(cols));   // rare: nothing of it is held in registers
#pragma unroll
      for (int b = 0; b < MBX; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) any |= 16 * b < rows && r < cols && y[b][r] == y[b][r];
      if (__ballot(any) == 0ull) top = 0xFFFFFFFFu;
    }
    if (lane == 0) red[p] = __builtin_bit_cast(float, top + 1u);   // 0: NaNs alone
    lds_barrier();   // and every wave has read this token's X
    top = __builtin_bit_cast(uint32_t, red[min(li, nb - 1)]);
    top = max(top, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0xB1, 0xF, 0xF, false));
    top = max(top, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0x4E, 0xF, 0xF, false));
    top = max(top, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0x141, 0xF, 0xF, false));
    top = max(top, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0x140, 0xF, 0xF, false));
    top = (uint32_t)__builtin_amdgcn_readfirstlane((int)top);
    const float s = top == 0u ? INFINITY : fq_scale_abs<F32T>(__builtin_bit_cast(float, top - 1u), clip);
    const int64_t t = g * d.tpb + tau;
    if (st == 0 && t < tokens) out_scales[t] = s;

    // Codes into the staging area, 4 columns (rem of them in the row) per row block.
    const float rcp = 1.0f / s;
    const bool plain = __builtin_amdgcn_readfirstlane((int)(s > 0.f && s < 1e37f && (__builtin_bit_cast(uint32_t, s) & 0x7FFFFFu) != 0x7FFFFFu)) != 0;
    int lane_at = li * N + 16 * p + 4 * lg;
    asm volatile("" : "+v"(lane_at));
    auto codes = [&](auto pk, auto&& word) __attribute__((always_inline)) {
      constexpr bool PK = decltype(pk)::value;
#pragma unroll
      for (int b = 0; b < MBX; ++b) {
        const uint32_t w = word(b);
        if (b >= MBX - 2 && 16 * b + li >= M) continue;
        const int at = lane_at + 16 * b * N;
        unsigned char* const o = cs + (PK ? at >> 1 : at);
        if ((N & 3) == 0) {
          if constexpr (PK) *reinterpret_cast<uint16_t*>(o) = (uint16_t)w;
          else *reinterpret_cast<uint32_t*>(o) = w;
        } else if constexpr (PK) {   // N even: a byte holds two columns of one row
#pragma unroll
          for (int k = 0; k < 2; ++k)
            if (2 * k + 2 <= rem) o[k] = (unsigned char)(w >> (8 * k));
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (k < rem) o[k] = (unsigned char)(w >> (8 * k));
        }
      }
    };
    constexpr std::true_type kPack;
    constexpr std::false_type kBytes;
    if (rem > 0) {
      if (plain && d.pack) codes(kPack, [&](int b) __attribute__((always_inline)) { return f32_codes4<true>(y[b], s, rcp); });
      else if (plain) codes(kBytes, [&](int b) __attribute__((always_inline)) { return f32_codes4<false>(y[b], s, rcp); });
      else {
#pragma unroll
        for (int b = 0; b < MBX; ++b) {
          uint32_t w = f32_codes4_div(y[b], s, d.pack != 0);
          int cols = 16 * b + li < M ? min(rem, 4) : 0, at = lane_at + 16 * b * N, step = d.pack ? 2 : 1;
          if (d.pack) at >>= 1;
          asm volatile("" : "+v"(w), "+v"(cols), "+v"(at));
          for (; cols > 0; cols -= step, w >>= 8) cs[at++] = (unsigned char)w;   // N even when packing
        }
      }
    }
    const int64_t gn = g + gridDim.x;
    const bool more = gn < ngroups;
    auto next_x = [&]() __attribute__((always_inline)) {
      if (!more) return;
      write_x();
      if (gn + gridDim.x < ngroups) load_x((gn + gridDim.x) * d.tpb + tau);
    };
    if (!d.alias) next_x();
    lds_barrier();   // the staged codes (and the next X) are whole
    if (t < tokens) {
      unsigned char* const o = reinterpret_cast<unsigned char*>(out_codes) + t * cbytes;
      if ((cbytes & 15) == 0) {
        for (int i = st; i < cbytes >> 4; i += nts) reinterpret_cast<v4i*>(o)[i] = reinterpret_cast<const v4i*>(cs)[i];
      } else {
        for (int i = st; i < cbytes >> 2; i += nts) reinterpret_cast<int*>(o)[i] = reinterpret_cast<const int*>(cs)[i];
      }
    }
    if (!more) break;
    if (d.alias) {
      lds_barrier();   // the codes have been read
      zero_pads();
      next_x();
      lds_barrier();
    }
    g = gn;
  }
}

template <int MBX, int KQX>
bool launch_f32_shape(const float* x, int64_t tokens, int64_t x_ld, const float* left, const float* right, int M,
                      int N, float clip, int pack, void* out_codes, float* out_scales, hipStream_t stream) {
  constexpr int kLds = 160 * 1024;
  const int cus = device_cu_count();
  FqF32 d{};
  d.M = M;
  d.N = N;
  d.F = M * N;
  d.mb = (M + 15) / 16;
  d.nb = (N + 15) / 16;
  d.pack = pack;
  // small widths: several tokens per workgroup, while two workgroups per CU remain
  d.tpb = (int)std::max<int64_t>(1, std::min<int64_t>(std::min(4, 8 / d.nb), tokens / (2 * cus)));
  d.inv_n = (uint32_t)(((1ull << 32) + N - 1) / N);
  d.px = 16 * d.nb + 4;
  d.xslot = 16 * d.mb * d.px * 4;
  d.cslot = ((pack ? d.F / 2 : d.F) + 15) / 16 * 16;
  const int waves = d.nb * d.tpb;
  const int red_bytes = d.tpb * 64;
  const int xbytes = d.tpb * d.xslot, cbytes = d.tpb * d.cslot;
  const int fixed = MBX * MBX * 1024 + red_bytes;
  const int most = std::max(1, 16 / waves);
  auto per_cu = [&](int area) { return std::min(most, kLds / (area + fixed)); };
  d.alias = per_cu(std::max(xbytes, cbytes)) > per_cu(xbytes + cbytes);
  d.stage_off = d.alias ? 0 : xbytes;
  const int area = (d.alias ? std::max(xbytes, cbytes) : xbytes + cbytes);
  d.lf_off = area;
  d.red_off = area + MBX * MBX * 1024;
  const int lds = d.red_off + red_bytes;
  if (lds > kLds) return false;
  auto kern = fq_f32_kernel<MBX, KQX>;
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return false;
  const int64_t ngroups = (tokens + d.tpb - 1) / d.tpb;
  const int64_t grid = std::min<int64_t>(ngroups, (int64_t)cus * std::max(1, per_cu(area)));
  launch(kern, dim3((unsigned)grid), dim3(64 * waves), (size_t)lds, stream, x, tokens, x_ld, left, right, d, clip,
         out_codes, out_scales);
  return true;
}

}  // namespace

// Launches fq_f32_kernel if it takes M x N and its LDS fits; false otherwise
// (nothing launched). Needs F % 8 == 0, clip > 0 and finite, x rows and the
// codes 16-byte aligned, N even when packing.
bool launch_f32(const float* x, int64_t tokens, int64_t x_ld, const float* left, const float* right, int M, int N,
                float clip, int pack, void* out_codes, float* out_scales, hipStream_t stream) {
  if (M < 2 || N < 2 || N > 256 || M > 128 || ((int64_t)M * N) % 8 != 0 || (pack && N % 2 != 0)) return false;
  const int mbx = (M + 31) / 32 * 2;
#define QO_F32(MBX_, KQX_)                                                                                         \
  if (mbx == MBX_ && N <= 16 * KQX_)                                                                               \
    return launch_f32_shape<MBX_, KQX_>(x, tokens, x_ld, left, right, M, N, clip, pack, out_codes, out_scales, stream);
#define QO_F32_ROWS(KQX_) QO_F32(2, KQX_) QO_F32(4, KQX_) QO_F32(6, KQX_) QO_F32(8, KQX_)
  QO_F32_ROWS(4)
  QO_F32_ROWS(8)
  QO_F32_ROWS(12)
  QO_F32_ROWS(16)
#undef QO_F32_ROWS
#undef QO_F32
  return false;
}

}  // namespace qo
