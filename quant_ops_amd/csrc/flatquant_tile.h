// Fused FlatQuant quantize for even widths up to 256 and heights up to 176
// (fp16 / bf16): fq_tile_kernel, the kernel behind the shapes without one of
// their own in flatquant_quant.hip. The loops' lengths are compile-time (MBX, KS:
// the shape rounded up to blocks of 32 rows and columns); M and N themselves are
// arguments, so 38 instances per type cover every even width and every height
// but the tall ones: M > 64 with N <= 32, M > 96 with N <= 64, M > 128 with
// N <= 96 and M > 160 with N <= 128 stay on the generic kernel, as do odd N,
// N > 256 and M > 176.
#pragma once

#include <algorithm>

#include "flatquant_common.h"

namespace qo {

// A launch's sizes and LDS plan (byte offsets). inv_n, inv_m: ceil(2^32 / N)
// and ceil(2^32 / M), for row = umulhi(e, inv), exact for e < 2^16.
struct FqTile {
  int M, N, F, mb, nb;   // mb = ceil(M / 16): MBX or one less; nb = ceil(N / 16): 2 KS or one less
  int tpb;               // token slots per workgroup
  uint32_t inv_n, inv_m;
  int x_off, xslot;      // X rows of slot 0; bytes of a slot
  int stage_off, cslot;  // staged codes of slot 0; bytes of a slot
  int alias;             // the codes are staged over X's rows
  int lf_off, red_off;   // L's fragments, the scale exchange
  int r_round, l_off;    // set-up: rows of R staged at a time; where L is staged beside the last ones (-1: by itself)
  int x_apart;           // X's rows lie outside the set-up's staging area
  int pack;
};

template <int MBX, int KS>
struct FqTileShape {
  static constexpr int KS2 = (MBX + 1) / 2;       // 32-deep slabs of the second product
  static constexpr int PX = 32 * KS + 8;          // X and R row pitch in elements: 16 rows start on 16 bank groups
  static constexpr int PL = 16 * MBX + 8;         // L row pitch while it is staged
  static constexpr int LF_BYTES = MBX * KS2 * 1024;
  static constexpr int L_BYTES = 32 * KS2 * PL * 2;
  static constexpr int XCH = (MBX + 1) / 2;       // 16-byte chunks per thread: X (M N / 8 over 64 nb threads)
  static constexpr int RCH = KS;                  // R
  static constexpr int LCH = (MBX * MBX + 4 * KS - 3) / (4 * KS - 2);   // L
  static constexpr int MAX_THREADS = KS <= 4 ? 512 : 128 * KS;
  // Waves per SIMD the registers are allocated for: what the threads (one
  // workgroup of 9 to 12 or 13 to 16 waves, or two of up to 8) and the LDS allow.
  // The price is spilled VGPRs in some instances (fp16, bf16 up to 6 fewer or, at
  // 10 x 7 and 11 x 7, up to 21): MBX x KS = 8 x 3 13, 8 x 4 17, 10 x 5 and 10 x 6 2
  // and 6, 11 x 5 and 11 x 6 25 and 29, 6 x 7 and 6 x 8 5 and 7, 8 x 7 and 8 x 8 32
  // and 38, 10 x 7 and 10 x 8 88 and 72, 11 x 7 and 11 x 8 129; and 14 to 52 SGPRs
  // (into VGPR lanes) in all of them.
  static constexpr int WAVES_PER_SIMD = KS <= 4 ? (MBX >= 10 ? 2 : 4) : KS <= 6 ? 3 : 4;
};

// Eight consecutive elements of a contiguous [rows, ncols] matrix into LDS rows
// of `pitch` elements, the first at `at`, column col, in pieces of G elements
// (ncols % G == 0).
template <int G, class T>
__device__ inline void fq_tile_put8(T* at, int col, int pitch, int ncols, v4i v) {
#pragma unroll
  for (int p = 0; p < 8 / G; ++p) {
    if constexpr (G == 8) *reinterpret_cast<v4i*>(at) = v;
    if constexpr (G == 4) *reinterpret_cast<v2i*>(at) = v2i{v[2 * p], v[2 * p + 1]};
    if constexpr (G == 2) *reinterpret_cast<int*>(at) = v[p];
    if constexpr (G == 1) *reinterpret_cast<short*>(at) = (short)((uint32_t)v[p >> 1] >> (16 * (p & 1)));
    at += G;
    col += G;
    if (G < 8 && col >= ncols) {
      col = 0;
      at += pitch - ncols;
    }
  }
}
// f(integral_constant<G>) for the largest piece that divides ncols (EVEN: ncols is even).
template <bool EVEN, class Fn>
__device__ __attribute__((always_inline)) inline void fq_tile_pieces(int ncols, Fn&& f) {
  if ((ncols & 7) == 0) f(std::integral_constant<int, 8>{});
  else if ((ncols & 3) == 0) f(std::integral_constant<int, 4>{});
  else if (EVEN || (ncols & 1) == 0) f(std::integral_constant<int, 2>{});
  else f(std::integral_constant<int, 1>{});
}

// The set-up's copy of L or R (a contiguous [rows, ncols] matrix, 16-byte
// aligned): CH chunks and one element of the tail per thread into registers,
// and from there the rows k0 .. k1 into LDS rows of `pitch` elements (k0 ncols a
// multiple of 8).
template <class T, int CH>
struct FqTileRows {
  v4i v[CH];
  T tail;
  __host__ __device__ void load(const T* __restrict__ src, int elems, int tid, int nt) {
    const int chunks = elems >> 3;
    if (chunks > 0) {   // a 2 x 2 matrix is all tail
#pragma unroll
      for (int i = 0; i < CH; ++i) v[i] = reinterpret_cast<const v4i*>(src)[min(tid + i * nt, chunks - 1)];
    }
    tail = src[min(8 * chunks + tid, elems - 1)];
  }
  template <bool EVEN>
  __device__ void put(T* dst, int pitch, int elems, int ncols, uint32_t inv, int k0, int k1, int tid, int nt) const {
    asm volatile("" : "+v"(tid));   // addresses computed here, not held across the set-up
    const int chunks = elems >> 3, e0 = k0 * ncols, e1 = min(k1 * ncols, elems);
    fq_tile_pieces<EVEN>(ncols, [&](auto gran) {
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int e = 8 * (tid + i * nt), row = (int)__umulhi((uint32_t)(e - e0), inv), col = e - e0 - row * ncols;
        if (tid + i * nt < chunks && e >= e0 && e < e1)
          fq_tile_put8<decltype(gran)::value>(dst + row * pitch + col, col, pitch, ncols, v[i]);
      }
    });
    const int e = 8 * chunks + tid;
    if (e >= e0 && e < e1) {
      const int row = (int)__umulhi((uint32_t)(e - e0), inv);
      dst[row * pitch + e - e0 - row * ncols] = tail;
    }
  }
};

// Four codes of one token row from yp (Y of columns n0 .. n0 + 3 as two D
// pairs), as four nibbles (code + 8) in bits 0 .. 15. rcp = 1 / s, finite. A NaN
// gives nibble 0, as the fallback's uint8 cast does.
template <class DT>
__device__ inline uint32_t fq_tile_nibbles(const uint32_t (&yp)[2], float rcp) {
  using Epi = FqEpi<DT>;
  if constexpr (std::is_same<DT, BF16T>::value) {
    float t[4];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(t[2 * r]) : "v"(__builtin_amdgcn_fmed3f(Epi::lo(yp[r]) * rcp, -8.0f, 7.0f)));
      asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(t[2 * r + 1]) : "v"(__builtin_amdgcn_fmed3f(Epi::hi(yp[r]) * rcp, -8.0f, 7.0f)));
    }
    const float magic = 12582920.0f;
    uint32_t ev, od;
    Epi::template code_byte<0, true>(ev, t[0], magic);
    Epi::template code_byte<0, true>(od, t[1], magic);
    Epi::template code_byte<1, false>(ev, t[2], magic);
    Epi::template code_byte<1, false>(od, t[3], magic);
    return ev | (od << 4);
  } else {
    uint32_t u[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const float a0 = __builtin_amdgcn_fmed3f(mul_f16lo(yp[r], rcp), -8.0f, 7.0f);
      const float a1 = __builtin_amdgcn_fmed3f(mul_f16hi(yp[r], rcp), -8.0f, 7.0f);
      const v2h magic = {(_Float16)1544.0f, (_Float16)1544.0f};   // FqEpi<F16T>::accumulate
      u[r] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, Epi::pack(a0, a1)) + magic) & 0x000F000Fu;
    }
    const uint32_t w = u[0] | (u[1] << 8);   // codes 0, 2 in the low half, 1, 3 in the high one
    return w | (w >> 12);
  }
}

// ---------------------------------------------------------------------------
// nb waves share a token, one per block p of 16 columns; small widths put tpb
// tokens into a workgroup. Rounding points are those of fq_mfma_kernel
// (flatquant_quant.hip), and so is the k order of both products.
//
// A wave per 16 columns instead of 32 reads every X and L operand from LDS
// twice as often per MFMA (1 KiB each, which the LDS still keeps up with) but
// halves the registers, so that four waves share a SIMD: one wave's codes and
// LDS reads run under another's MFMAs.
//
// X: a token is contiguous in memory, so it is read as whole 16-byte pieces
// whatever its row length, one token ahead into registers, and written to LDS
// rows of PX elements (in 16-, 8- or 4-byte pieces), where an operand is one
// conflict-free 16-byte read. Padding (rows M .. 16 mb, columns N .. 32 KS) is
// zeroed once and never written again. R's fragments are in VGPRs, L's in LDS.
//
// Codes are staged in LDS in memory order and leave as whole 16-byte pieces
// while the next token's first product runs (two barriers per token; four where
// they are staged over X's rows to let a second workgroup share the CU).
//
// Bound: no unit alone (128 x 148, 4096 tokens: LDS 46 %, VALU 39 %, MFMA 25 %
// busy), the barriers between a token's phases at 2.5 to 3 waves per SIMD.
// Measured (same box, kernel alone, before: fq_generic_kernel for 96 x 96,
// fq_mfma_kernel's 4-byte copies or zero-padded fragments for the others):
//   fp16  777 x  96 x  96 int8    110 -> 15.8 us
//   bf16 1021 x 128 x 148          44 -> 25.7 us,  4096 tokens 138 -> 88 us
//   bf16 1021 x  86 x 128          25 -> 17.5 us,  1021 x 108 x 128  31 -> 22 us
//   bf16 4096 x 144 x 192         146 -> 125 us (2.3 TB/s), 16 x 64 x 214  13.5 -> 10.3 us
// A wave per 32 columns (half the LDS reads, 230 registers, one wave per SIMD)
// took 137 us at 4096 x 128 x 148; 96 registers for two workgroups of ten waves
// spill 76 of them.
// ---------------------------------------------------------------------------
template <class DT, int MBX, int KS>
__global__ void __launch_bounds__((FqTileShape<MBX, KS>::MAX_THREADS)) __attribute__((amdgpu_waves_per_eu(FqTileShape<MBX, KS>::WAVES_PER_SIMD)))
fq_tile_kernel(const typename DT::T* __restrict__ x, int64_t tokens, int64_t x_ld,
               const typename DT::T* __restrict__ left, const typename DT::T* __restrict__ right, FqTile d, float clip,
               void* __restrict__ out_codes, float* __restrict__ out_scales) {
  using S = FqTileShape<MBX, KS>;
  using T = typename DT::T;
  using Ops = MfmaOps<DT>;
  using V = typename Ops::V;
  using Epi = FqEpi<DT>;
  constexpr int KS2 = S::KS2, PX = S::PX, PL = S::PL;

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
  const int M = d.M, N = d.N, F = d.F;
  T* const xs = reinterpret_cast<T*>(smem + d.x_off + tau * d.xslot);
  unsigned char* const cs = smem + d.stage_off + tau * d.cslot;
  float* const red = reinterpret_cast<float*>(smem + d.red_off) + tau * 16;
  const int64_t ngroups = (tokens + d.tpb - 1) / d.tpb;

  // One token into registers, at most XCH chunks of 8 elements per thread, and
  // from there into its rows: chunk i at element offset xat[i] >> 8 of xs,
  // column xat[i] & 255 (N <= 256).
  const int nch = F >> 3;
  v4i xr[S::XCH];
  uint32_t xat[S::XCH];
#pragma unroll
  for (int i = 0; i < S::XCH; ++i) {
    const uint32_t e = 8 * (st + i * nts), row = __umulhi(e, d.inv_n), col = e - row * N;
    xat[i] = (row * PX + col) << 8 | col;
  }
  auto load_x = [&](int64_t t) __attribute__((always_inline)) {
    const char* src = reinterpret_cast<const char*>(x + (t < tokens ? t : tokens - 1) * x_ld);
#pragma unroll
    for (int i = 0; i < S::XCH; ++i) xr[i] = *reinterpret_cast<const v4i*>(src + 16u * (uint32_t)min(st + i * nts, nch - 1));
  };
  auto write_x = [&]() __attribute__((always_inline)) {
    fq_tile_pieces<true>(N, [&](auto gran) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < S::XCH; ++i)
        if (st + i * nts < nch)
          fq_tile_put8<decltype(gran)::value>(xs + (xat[i] >> 8), (int)(xat[i] & 255u), PX, N, xr[i]);
    });
  };
  auto zero_pads = [&]() __attribute__((always_inline)) {
    for (int r = st; r < M; r += nts)
      for (int c = N; c < 32 * KS; c += 2) *reinterpret_cast<int*>(xs + r * PX + c) = 0;
    for (int i = st; i < (16 * d.mb - M) * (PX / 8); i += nts) reinterpret_cast<v4i*>(xs + M * PX)[i] = v4i{0, 0, 0, 0};
  };

  int64_t g = blockIdx.x;   // grid <= ngroups
  V rf[KS];
  {
    // Set-up: R, L and the first token requested together. R goes row-major
    // through LDS, r_round rows at a time, into B operands of the first product:
    // rf[ks][j] = R[32ks + 8lg + j][16p + li], 0 in the padding, by LDS transpose
    // reads (rows past the staged ones read stale LDS, then masked).
    FqTileRows<T, S::RCH> rr;
    FqTileRows<T, S::LCH> lr;
    rr.load(right, N * N, tid, nt);
    lr.load(left, M * M, tid, nt);
    load_x(g * d.tpb + tau);
    T* const rst = reinterpret_cast<T*>(smem);
    T* const lst = reinterpret_cast<T*>(smem + max(d.l_off, 0));
    if (d.x_apart) zero_pads();
#pragma unroll 1
    for (int k0 = 0; k0 < 32 * KS; k0 += d.r_round) {
      if (k0 > 0) lds_barrier();
      rr.template put<true>(rst, PX, N * N, N, d.inv_n, k0, k0 + d.r_round, tid, nt);
      if (k0 + d.r_round >= 32 * KS) {
        if (d.l_off >= 0) lr.template put<false>(lst, PL, M * M, M, d.inv_m, 0, M, tid, nt);
        if (d.x_apart) write_x();
      }
      lds_barrier();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (32 * ks < k0 || 32 * ks >= k0 + d.r_round) continue;
        const T* at = rst + (32 * ks - k0 + 8 * lg + (li >> 2)) * PX + 16 * p + 4 * (li & 3);
        V v = join_tr16<V>(lds_tr16(at), lds_tr16(at + 4 * PX));
        if (ks == KS - 1) {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (32 * ks + 8 * lg + j >= N) v[j] = DT::from_f(0.0f);
        }
        rf[ks] = 16 * p + li < N ? v : V{};
      }
    }
    if (d.l_off < 0) {
      lds_barrier();
      lr.template put<false>(lst, PL, M * M, M, d.inv_m, 0, M, tid, nt);
      lds_barrier();
    }
    // L's fragments, split over the waves: element j of (b, s) is L[m'][16b + li],
    // m' = 32s + 16(j/4) + 4lg + j%4 (the row order of Z's accumulator pairs)
#pragma unroll 1
    for (int f = wave; f < MBX * KS2; f += nt >> 6) {
      const int b = f / KS2, s = f % KS2;
      const T* at = lst + (32 * s + 4 * lg + (li >> 2)) * PL + 16 * b + 4 * (li & 3);
      V v = join_tr16<V>(lds_tr16(at), lds_tr16(at + 16 * PL));
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (16 * b + li >= M || 32 * s + 16 * (j >> 2) + 4 * lg + (j & 3) >= M) v[j] = DT::from_f(0.0f);
      *reinterpret_cast<V*>(lf + f * 1024 + 16 * lane) = v;
    }
    lds_barrier();
  }
  if (!d.x_apart) {
    zero_pads();
    write_x();
    lds_barrier();
  }
  if (g + gridDim.x < ngroups) load_x((g + gridDim.x) * d.tpb + tau);

  const T* const xa = xs + li * PX + 8 * lg;       // A operand (rb, ks) at (16 rb) PX + 32 ks
  const int rem = N - (16 * p + 4 * lg);           // this lane's columns inside the row (4 or more: all)
  const int cbytes = d.pack ? F >> 1 : F;
  const bool full = d.mb == MBX;
  // Rows of the last two row blocks inside the token, as masks of D pairs: a
  // padded row of Z is 0 whatever R holds.
  uint32_t zmask[2][2];
#pragma unroll
  for (int e = 0; e < 2; ++e)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int m = 16 * (MBX - 2 + e) + 4 * lg + 2 * h;
      zmask[e][h] = (m < M ? 0xFFFFu : 0u) | (m + 1 < M ? 0xFFFF0000u : 0u);
    }
  while (true) {
    // First product, rounding point 1, accumulators -> A operands of the
    // second: zp[s][4e + r] = Z[32s + 16e + 4lg + r][16p + li].
    V zp[KS2];
#pragma unroll
    for (int s = 0; s < KS2; ++s) {
      v4f c[2] = {};
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int rb = 2 * s + e;
        if (rb >= MBX || (rb == MBX - 1 && !full)) continue;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          c[e] = Ops::mfma(*reinterpret_cast<const V*>(xa + 16 * rb * PX + 32 * ks), rf[ks], c[e]);
      }
      v4i z;
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int rb = 2 * s + e;
          const uint32_t v = Epi::pack_acc(c[e][2 * h], c[e][2 * h + 1]);
          z[2 * e + h] = rb >= MBX ? 0 : (int)(rb >= MBX - 2 ? v & zmask[rb - (MBX - 2)][h] : v);
        }
      zp[s] = __builtin_bit_cast(V, z);
      __builtin_amdgcn_sched_barrier(0);   // or every slab's reads are hoisted and spill
    }

    // Second product, transposed, rounding point 2: yp[b] = Y[16b + li][16p + 4lg .. + 3].
    // max |Y| of the raw accumulators (rounding is monotonic); the padding's are
    // 0, or NaN, which fmaxf drops.
    uint32_t yp[MBX][2];
    float amax = 0.f;
#pragma unroll
    for (int b = 0; b < MBX; ++b) {
      if (b == MBX - 1 && !full) continue;
      v4f c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS2; ++s)
        c = Ops::mfma(zp[s], *reinterpret_cast<const V*>(lf + (b * KS2 + s) * 1024 + 16 * lane), c);
      amax = fmaxf(fmaxf(amax, fabsf(c[0])), fabsf(c[1]));
      amax = fmaxf(fmaxf(amax, fabsf(c[2])), fabsf(c[3]));
      yp[b][0] = Epi::pack_acc(c[0], c[1]);
      yp[b][1] = Epi::pack_acc(c[2], c[3]);
      if (b % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
    auto y_at = [&](int b, int r) __attribute__((always_inline)) { return r & 1 ? Epi::hi(yp[b][r >> 1]) : Epi::lo(yp[b][r >> 1]); };
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
        for (int r = 0; r < 4; ++r) any |= 16 * b < rows && r < cols && (b < MBX - 1 || full) && y_at(b, r) == y_at(b, r);
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
    const float s = top == 0u ? INFINITY : fq_scale_abs<DT>(DT::round(__builtin_bit_cast(float, top - 1u)), clip);
    const int64_t t = g * d.tpb + tau;
    if (st == 0 && t < tokens) out_scales[t] = s;

    // Codes into the staging area, 4 columns (rem of them in the row) per row
    // block: nibbles (16 bits at nibble m N + 16p + 4lg, an even one) or bytes.
    const float rcp = 1.0f / s;
    const bool plain = __builtin_amdgcn_readfirstlane((int)(s > 0.f && s < INFINITY)) != 0;
    int lane_at = li * N + 16 * p + 4 * lg;
    asm volatile("" : "+v"(lane_at));   // offsets computed per token instead of held in VGPRs
    // G: 4 where N % 4 == 0 (whole stores), else 2
    auto codes = [&](auto pk, auto gran, auto&& word) __attribute__((always_inline)) {
      constexpr bool PK = decltype(pk)::value;
      constexpr int G = decltype(gran)::value;
#pragma unroll
      for (int b = 0; b < MBX; ++b) {
        if (b == MBX - 1 && !full) continue;
        const uint32_t w = word(b);
        if (b >= MBX - 2 && 16 * b + li >= M) continue;
        const int at = lane_at + 16 * b * N;
        unsigned char* const o = cs + (PK ? at >> 1 : at);
        if constexpr (PK && G == 4) *reinterpret_cast<uint16_t*>(o) = (uint16_t)w;
        if constexpr (!PK && G == 4) *reinterpret_cast<uint32_t*>(o) = w;
        if constexpr (PK && G == 2) {
          o[0] = (unsigned char)w;
          if (rem >= 4) o[1] = (unsigned char)(w >> 8);
        }
        if constexpr (!PK && G == 2) {
          reinterpret_cast<uint16_t*>(o)[0] = (uint16_t)w;
          if (rem >= 4) reinterpret_cast<uint16_t*>(o)[1] = (uint16_t)(w >> 16);
        }
      }
    };
    auto nibbles = [&](int b) __attribute__((always_inline)) { return fq_tile_nibbles<DT>(yp[b], rcp); };
    auto bytes = [&](int b) __attribute__((always_inline)) {
      uint32_t w = 0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float y = y_at(b, r);
        const int code = (int)__builtin_rintf(DT::round(__builtin_amdgcn_fmed3f(y * rcp, -8.0f, 7.0f)));
        w |= (uint32_t)((y != y ? 0 : code) & 0xFF) << (8 * r);
      }
      return w;
    };
    auto slow_nibbles = [&](int b) __attribute__((always_inline)) {
      uint32_t w = 0;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        w |= (uint32_t)(fq_code_from_quot<true>(DT::round(opaque(y_at(b, r)) / s)) + 8) << (4 * r);
      __builtin_amdgcn_sched_barrier(0);
      return w;
    };
    auto slow_bytes = [&](int b) __attribute__((always_inline)) {
      uint32_t w = 0;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        w |= (uint32_t)(fq_code_from_quot<false>(DT::round(opaque(y_at(b, r)) / s)) & 0xFF) << (8 * r);
      __builtin_amdgcn_sched_barrier(0);
      return w;
    };
    constexpr std::true_type kPack;
    constexpr std::false_type kBytes;
    constexpr std::integral_constant<int, 4> k4;
    constexpr std::integral_constant<int, 2> k2;
    if (rem > 0) {
      const bool four = (N & 3) == 0;
      if (plain && d.pack) {
        if (four) codes(kPack, k4, nibbles);
        else codes(kPack, k2, nibbles);
      } else if (plain) {
        if (four) codes(kBytes, k4, bytes);
        else codes(kBytes, k2, bytes);
      } else if (d.pack) {   // a scale of 0 or infinity: the fallback's quotients
        if (four) codes(kPack, k4, slow_nibbles);
        else codes(kPack, k2, slow_nibbles);
      } else {
        if (four) codes(kBytes, k4, slow_bytes);
        else codes(kBytes, k2, slow_bytes);
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

// Launches the instance for M x N if there is one and its LDS fits; false
// otherwise (nothing launched). Needs F % 8 == 0, clip > 0 and finite, x rows,
// L, R and the codes 16-byte aligned.
template <class DT, int MBX, int KS>
static bool launch_tile_shape(const void* x, int64_t tokens, int64_t x_ld, const void* left, const void* right, int M,
                              int N, float clip, int pack, void* out_codes, float* out_scales, hipStream_t stream) {
  using S = FqTileShape<MBX, KS>;
  using T = typename DT::T;
  constexpr int kLds = 160 * 1024;
  const int cus = device_cu_count();
  FqTile d{};
  d.M = M;
  d.N = N;
  d.F = M * N;
  d.mb = (M + 15) / 16;
  d.nb = (N + 15) / 16;
  d.pack = pack;
  // small widths: several tokens per workgroup, while two workgroups per CU remain
  d.tpb = (int)std::max<int64_t>(1, std::min<int64_t>(std::min(4, 8 / d.nb), tokens / (2 * cus)));
  d.inv_n = (uint32_t)(((1ull << 32) + N - 1) / N);
  d.inv_m = (uint32_t)(((1ull << 32) + M - 1) / M);
  d.xslot = 16 * d.mb * S::PX * 2;
  d.cslot = ((pack ? d.F / 2 : d.F) + 15) / 16 * 16;
  const int waves = d.nb * d.tpb;
  const int red_bytes = d.tpb * 64;
  const int row = S::PX * 2;
  const int xbytes = d.tpb * d.xslot, cbytes = d.tpb * d.cslot;
  const int fixed = S::LF_BYTES + red_bytes + 64;
  const int stage_all = 32 * KS * row + S::L_BYTES;   // R's and L's rows at once
  const int stage_min = std::max(32 * row, S::L_BYTES);
  const int most = std::max(1, 16 / waves);           // four waves per SIMD
  auto per_cu = [&](int area) { return std::min(most, kLds / (area + fixed)); };
  const int64_t ngroups = (tokens + d.tpb - 1) / d.tpb;
  const int64_t wanted = std::min<int64_t>(most, (ngroups + cus - 1) / cus);   // workgroups per CU
  int area;
  if (per_cu(stage_all + xbytes + cbytes) >= wanted) {
    // nothing shares its place
    d.x_apart = 1;
    d.x_off = stage_all;
    d.stage_off = d.x_off + xbytes;
    area = d.stage_off + cbytes;
    d.r_round = 32 * KS;
    d.l_off = 32 * KS * row;
  } else {
    // staging in the area of X and the codes; the codes over X where that lets
    // one more workgroup onto the CU
    const int apart = std::max(xbytes + cbytes, stage_min), over = std::max({xbytes, cbytes, stage_min});
    d.alias = per_cu(over) > per_cu(apart);
    area = d.alias ? over : apart;
    d.x_off = 0;
    d.stage_off = d.alias ? 0 : xbytes;
    if (area < stage_all && per_cu(stage_all) == per_cu(area)) area = stage_all;
    area = (area + 15) / 16 * 16;
    d.r_round = std::min(32 * KS, area / row / 32 * 32);
    const int last = (32 * KS - 1) / d.r_round * d.r_round;   // first row of the last round
    const int l_at = (32 * KS - last) * row;
    d.l_off = l_at + S::L_BYTES <= area ? l_at : -1;
  }
  d.lf_off = area;
  d.red_off = area + S::LF_BYTES;
  const int lds = d.red_off + red_bytes;
  if (lds > kLds) return false;
  auto kern = fq_tile_kernel<DT, MBX, KS>;
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return false;
  const int64_t grid = std::min<int64_t>(ngroups, (int64_t)cus * std::max(1, per_cu(area)));
  launch(kern, dim3((unsigned)grid), dim3(64 * waves), (size_t)lds, stream, reinterpret_cast<const T*>(x), tokens,
         x_ld, reinterpret_cast<const T*>(left), reinterpret_cast<const T*>(right), d, clip, out_codes, out_scales);
  return true;
}

template <class DT>
bool launch_tile(const void* x, int64_t tokens, int64_t x_ld, const void* left, const void* right, int M, int N,
                 float clip, int pack, void* out_codes, float* out_scales, hipStream_t stream);

// Body of launch_tile, instantiated once per element type in a source of its own.
template <class DT>
static bool launch_tile_any(const void* x, int64_t tokens, int64_t x_ld, const void* left, const void* right, int M,
                            int N, float clip, int pack, void* out_codes, float* out_scales, hipStream_t stream) {
  if (M < 2 || N < 2 || N % 2 != 0 || N > 256 || M > 176 || ((int64_t)M * N) % 8 != 0) return false;
  const int ks = (N + 31) / 32;
  const int mbx = M > 160 ? 11 : (M + 31) / 32 * 2;
#define QO_TILE(MBX_, KS_)                                                                                          \
  if (mbx == MBX_ && ks == KS_)                                                                                     \
    return launch_tile_shape<DT, MBX_, KS_>(x, tokens, x_ld, left, right, M, N, clip, pack, out_codes, out_scales, \
                                            stream);
#define QO_TILE_ROWS(KS_) QO_TILE(2, KS_) QO_TILE(4, KS_) QO_TILE(6, KS_) QO_TILE(8, KS_) QO_TILE(10, KS_) QO_TILE(11, KS_)
  QO_TILE(2, 1) QO_TILE(4, 1)
  QO_TILE(2, 2) QO_TILE(4, 2) QO_TILE(6, 2)
  QO_TILE(2, 3) QO_TILE(4, 3) QO_TILE(6, 3) QO_TILE(8, 3)
  QO_TILE(2, 4) QO_TILE(4, 4) QO_TILE(6, 4) QO_TILE(8, 4) QO_TILE(10, 4)
  QO_TILE_ROWS(5)
  QO_TILE_ROWS(6)
  QO_TILE_ROWS(7)
  QO_TILE_ROWS(8)
#undef QO_TILE_ROWS
#undef QO_TILE
  return false;
}

}  // namespace qo
