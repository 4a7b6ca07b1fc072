// Fused dequantization + rotation back of the rotated backend
// (fade/rotated_quant.py:134-145,176-187) for fp16 / bf16 output and head_dim 128:
// out = x_rot @ R with x_rot = dtype(code * scale), read from the packed codes
// and written once.
//
// The two-step path moves x_rot through HBM four times (dequantized rows, an
// fp32 copy, the fp32 product, the 16-bit copy): 175 us for 33 M elements, of
// which the fp32 GEMM takes 95.  Here the codes are dequantized in registers
// into MFMA operands (one rounding to the output type, the reference's) and
// the product runs on the 16-bit matrix cores with R in three pieces of its
// type, which hold the 24 bits of every entry: bf16 as it is, fp16 at a
// power-of-two scale that puts max|R| in [2^14, 2^15) (entries below 2^-15 of the
// largest then end at 2^-39 of it).  Every product accumulates in fp32, the small
// pieces' first, so that their sums are not rounded at the result's size.
// Against 64 bits, 16 M outputs of each width and axis: as close as the fp32 GEMM or
// closer (4-bit fp16 9.2 k outputs not the nearest, the GEMM 20 k).  Two pieces in fp16 take
// 26 us of 31 for 33 M elements, but miss the last bit of 18% of the entries of an
// orthogonal R, and their 2-bit outputs were further off than the GEMM's.
//
// MFMA (32x32x16): C^T[out channel][row] = (R^T)[out][in] x_rot^T[in][row].
// Lane (n, h) of the B operand holds row n, input channels 64 h + 8 ks ..+ 7
// at step ks: the 64 channels of one lane are contiguous code bytes.  The
// order within every 8 channels is the one the code conversion produces; R^T
// is stored in LDS in that order, and its rows so that lane (n, h) receives
// the 16 consecutive output channels 32 mt + 16 h ..+ 15 of row n.
//
// One workgroup of 16 waves per CU: R's pieces and the output stage fill its LDS,
// and four waves per SIMD let one's conversions run under another's MFMAs.
// Measured (4-bit fp16, per call): 7.7 M elements 12.6 us, 33 M 31 (2.6 TB/s; the two-step
// path: 168 us), 66 M 56, 131 M 115.  The MFMAs and the reads of R's fragments from LDS,
// which take as long, bound it with the split of R in the prologue (7 us of a small
// call); two row tiles per wave, which share each fragment, took the same time
// (33 M 32.5, 66 M 56, 131 M 115).
#include <type_traits>

#include "fade_common.h"

namespace fade {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kD = 128;
constexpr int kWaves = 16;
constexpr int kThreads = 64 * kWaves;
constexpr int kRows = 32;     // rows of a wave's work item
constexpr int kPieces = 3;    // 16-bit pieces of R
constexpr int kRPitch = 136;  // halves per R^T row in LDS: 16-byte reads of 8 rows hit distinct banks
constexpr int kStagePitch = 80;  // bytes per staged row of 32 output channels (64 bytes): likewise

// Channel (within its group of 8) that slot e of an operand holds: the order
// in which dequant8 produces the codes of BITS.
template <int BITS>
__device__ constexpr int slot_channel(int e) {
  return BITS == 4 ? ((e & 1) << 2) + ((e >> 2) << 1) + ((e & 2) ? 0 : 1)  // 1 5 0 4 3 7 2 6
         : BITS == 2 ? ((e & 1) << 2) + (e >> 1)                            // 0 4 1 5 2 6 3 7
                     : e;
}
template <int BITS>
constexpr int kLaneBytes = BITS == 3 ? 64 : 8 * BITS;  // code bytes of 64 channels (3-bit codes are raw int8)

// Code bytes of one lane's 64 channels.
template <int BITS>
struct Codes {
  u32x4 w[kLaneBytes<BITS> / 16];
};

// The codes of 8 channels (group ks of the lane's 64) as four fp16 pairs, exact.
template <int BITS>
__device__ __forceinline__ void codes8(const Codes<BITS>& cd, int ks, f16x2 (&c)[4]) {
  if constexpr (BITS == 4) {
    // nibble -> mantissa bits 4..7 of 64.0 with its top bit flipped: 72 + c
    const uint32_t w = cd.w[ks >> 2][ks & 3];
    const uint32_t o[4] = {((w << 4) & 0x00F000F0u) ^ 0x54805480u, (w & 0x00F000F0u) ^ 0x54805480u,
                           ((w >> 4) & 0x00F000F0u) ^ 0x54805480u, ((w >> 8) & 0x00F000F0u) ^ 0x54805480u};
    const f16x2 k72 = {static_cast<_Float16>(72.0f), static_cast<_Float16>(72.0f)};
#pragma unroll
    for (int j = 0; j < 4; ++j) c[j] = __builtin_bit_cast(f16x2, o[j]) - k72;
  } else if constexpr (BITS == 2) {
    // two code bytes, one per half; a code -> mantissa bits 8..9 of 4.0 with its top bit flipped: 6 + c
    const uint32_t d = cd.w[0][ks >> 1];
    const uint32_t t = __builtin_amdgcn_perm(d, d, (ks & 1) ? 0x0C030C02u : 0x0C010C00u);
    const f16x2 k6 = {static_cast<_Float16>(6.0f), static_cast<_Float16>(6.0f)};
#pragma unroll
    for (int j = 0; j < 4; ++j)
      c[j] = __builtin_bit_cast(f16x2, ((t << (2 + 2 * j)) & 0x03000300u) ^ 0x46004600u) - k6;
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t d = cd.w[ks >> 1][2 * (ks & 1) + (j >> 1)] >> (16 * (j & 1));
      c[j] = f16x2{static_cast<_Float16>(static_cast<float>(static_cast<int8_t>(d & 0xFFu))),
                   static_cast<_Float16>(static_cast<float>(static_cast<int8_t>((d >> 8) & 0xFFu)))};
    }
  }
}

// dtype(code * scale) for the pairs of codes8; s: the scales of each pair
// (16-bit patterns, low half first).  fp16: one packed multiply, rounded once.
// bf16: the product of a small integer and 8 bits is exact in fp32.
template <bool BF>
__device__ __forceinline__ uint32_t scaled(f16x2 c, uint32_t s) {
#pragma clang fp contract(off)
  if constexpr (BF)
    return pack_bf16(static_cast<float>(c.x) * __uint_as_float(s << 16),
                     static_cast<float>(c.y) * __uint_as_float(s & 0xFFFF0000u));
  else
    return __builtin_bit_cast(uint32_t, c * __builtin_bit_cast(f16x2, s));
}

template <bool BF>
__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (BF)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// A scale whose products with the codes may not be finite: |s| >= 8192 (fp16) or
// 2^125 (bf16), inf and NaN among them.
template <bool BF>
__device__ __forceinline__ bool big_scale(uint32_t bits) { return (bits & 0x7FFFu) >= (BF ? 0x7E00u : 0x7000u); }

// The 16-bit values that are inf or NaN replaced by 0.
template <bool BF>
__device__ __forceinline__ u32x4 finite_only(u32x4 v) {
  constexpr uint32_t kExp = BF ? 0x7F80u : 0x7C00u;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if ((v[j] & kExp) == kExp) v[j] &= 0xFFFF0000u;
    if (((v[j] >> 16) & kExp) == kExp) v[j] &= 0x0000FFFFu;
  }
  return v;
}

// The next 16-bit piece of a value of R; a keeps the rest.  ANY: a value that is not
// finite is one piece, and one that rounds to the type's inf starts with its largest.
template <bool BF, bool ANY>
__device__ __forceinline__ uint32_t piece(float& a) {
  uint16_t p = f2w<BF>(a);
  if constexpr (ANY) {
    const bool finite = fabsf(a) < INFINITY;
    if (finite && (p & 0x7FFFu) == (BF ? 0x7F80u : 0x7C00u)) --p;
    a = finite ? a - w2f<BF>(p) : 0.0f;
  } else {
    a -= w2f<BF>(p);
  }
  return p;
}

// Work item `it` of a wave: 32 rows of one (b, h) slice (per-channel scales),
// or of the flattened rows (per-token scales: one slice).
template <int BITS, bool BF, bool TOKEN>
__global__ __launch_bounds__(kThreads) void rotdq_kernel(const uint8_t* __restrict__ packed,
                                                         const uint16_t* __restrict__ scale, int64_t S,
                                                         uint32_t blocks, uint32_t items, const float* __restrict__ R,
                                                         uint16_t* __restrict__ out) {
  constexpr int LB = kLaneBytes<BITS>;
  constexpr int RB = 2 * LB;  // bytes per packed row
  __shared__ __attribute__((aligned(16))) uint16_t rt[kPieces][kD][kRPitch];
  __shared__ __attribute__((aligned(16))) uint8_t stage[kWaves][kRows * kStagePitch];
  __shared__ float red[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- R^T in pieces into LDS: a thread turns the 2 x 4 blocks of two input
  // channels in neighbouring slots and four output channels, one dword per
  // output channel and piece.  A wave's 16 slot pairs x 4 channel quads put
  // two lanes on a bank (2-byte writes of one row at a time put eight) ----
  float unscale = 1.0f;
  {
    constexpr int kBlocks = kD / 2 * kD / 4 / kThreads;  // 2 x 4 blocks per thread
    float4 ra[kBlocks], rb[kBlocks];
    const int pair = tid & 15, quad = (tid >> 4) & 3, rest = tid >> 6;
    auto bits = [](float v) { return __float_as_uint(v) & 0x7FFFFFFFu; };  // of magnitudes, which order as they do
    uint32_t top = 0;
    // block i: slots 2 pp, 2 pp + 1 (pp = pair + 16 (k & 3)), output channels 4 (quad + 4 (k >> 2)) ..+ 3
#pragma unroll
    for (int i = 0; i < kBlocks; ++i) {
      const int k = rest + i * kWaves, pp = pair + 16 * (k & 3), e = 2 * (pp & 3), j0 = 4 * (quad + 4 * (k >> 2));
      const float* src = R + (8 * (pp >> 2)) * kD + j0;
      ra[i] = *reinterpret_cast<const float4*>(src + slot_channel<BITS>(e) * kD);
      rb[i] = *reinterpret_cast<const float4*>(src + slot_channel<BITS>(e + 1) * kD);
      for (const float v : {ra[i].x, ra[i].y, ra[i].z, ra[i].w, rb[i].x, rb[i].y, rb[i].z, rb[i].w}) top = max(top, bits(v));
    }
    // entries that are inf, NaN or round to a bf16 inf: rare, and split with more care
    const bool extreme = __builtin_amdgcn_ballot_w64(top >= (BF ? 0x7F7F8000u : 0x7F800000u)) != 0;
    float scale_r = 1.0f;
    if constexpr (!BF) {
      float mx = __uint_as_float(top);
      if (extreme) {  // the largest finite entry
        mx = 0.0f;
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
          for (const float v : {ra[i].x, ra[i].y, ra[i].z, ra[i].w, rb[i].x, rb[i].y, rb[i].z, rb[i].w})
            mx = bits(v) < 0x7F800000u ? fmaxf(mx, fabsf(v)) : mx;
      }
      mx = group_max<64>(mx);
      if (lane == 0) red[wave] = mx;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, red[w]);
      // 2^e with max|R| 2^e in [2^14, 2^15) (the largest finite entry); an orthogonal R's is at most 1
      const int e = mx > 0.0f ? 14 - ilogbf(mx) : 0;
      const int ec = e > 120 ? 120 : e;  // both powers are normal floats
      scale_r = ldexpf(1.0f, ec);
      unscale = ldexpf(1.0f, -ec);
    }
    auto split = [&](auto any) {
#pragma unroll
      for (int i = 0; i < kBlocks; ++i) {
        const int k = rest + i * kWaves, pp = pair + 16 * (k & 3), j0 = 4 * (quad + 4 * (k >> 2));
        const float fa[4] = {ra[i].x, ra[i].y, ra[i].z, ra[i].w}, fb[4] = {rb[i].x, rb[i].y, rb[i].z, rb[i].w};
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          // output channel 32 mt + 16 h' + 4 a + b sits in A row 32 mt + 8 a + 4 h' + b
          const int j = j0 + jj, row = (j & ~31) | (((j >> 2) & 3) << 3) | (((j >> 4) & 1) << 2) | (j & 3);
          float a = fa[jj] * scale_r, b = fb[jj] * scale_r;
#pragma unroll
          for (int q = 0; q < kPieces; ++q) {
            const uint32_t pa = piece<BF, decltype(any)::value>(a), pb = piece<BF, decltype(any)::value>(b);
            *reinterpret_cast<uint32_t*>(&rt[q][row][2 * pp]) = pa | (pb << 16);
          }
        }
      }
    };
    if (__builtin_expect(extreme, 0)) split(std::true_type{});
    else split(std::false_type{});
  }
  __syncthreads();

  auto rows_of = [&](uint32_t it, int64_t& slice, int64_t& r0) {  // the wave's first row of item it
    const uint32_t sl = TOKEN ? 0u : it / blocks;
    slice = sl;
    r0 = static_cast<int64_t>(it - sl * blocks) * kRows;
  };
  auto load = [&](uint32_t it, Codes<BITS>& cd, uint32_t& ts) {
    int64_t slice, r0;
    rows_of(it, slice, r0);
    const int64_t row = slice * S + (r0 + n < S ? r0 + n : S - 1);  // rows past the slice: its last row, never stored
    const u32x4* src = reinterpret_cast<const u32x4*>(packed + row * RB + h * LB);
#pragma unroll
    for (int k = 0; k < LB / 16; ++k) cd.w[k] = src[k];
    ts = TOKEN ? scale[row] : 0u;
  };

  // neighbouring items go to different workgroups, so a few of them spread over the CUs
  for (uint32_t it = wave * gridDim.x + blockIdx.x; it < items; it += kWaves * gridDim.x) {
    Codes<BITS> cd;
    uint32_t ts;
    load(it, cd, ts);
    __asm__ volatile("" ::: "memory");  // keep the R fragment reads inside the loop
    int64_t slice, r0;
    rows_of(it, slice, r0);
    u32x4 x[8];
    bool big = false;
    if constexpr (TOKEN) {
      const uint32_t s2 = ts | (ts << 16);
      big = big_scale<BF>(ts);
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        f16x2 c[4];
        codes8<BITS>(cd, ks, c);
#pragma unroll
        for (int j = 0; j < 4; ++j) x[ks][j] = scaled<BF>(c[j], s2);
      }
    } else {
      const u32x4* sp = reinterpret_cast<const u32x4*>(scale + slice * kD + 64 * h);
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        const u32x4 sw = sp[ks];
        uint32_t sv[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          sv[j] = (sw[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
          big |= big_scale<BF>(sv[j]);
        }
        f16x2 c[4];
        codes8<BITS>(cd, ks, c);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          x[ks][j] = scaled<BF>(c[j], sv[slot_channel<BITS>(2 * j)] | (sv[slot_channel<BITS>(2 * j + 1)] << 16));
      }
    }
    // inf times a piece of R of either sign would give NaN where the whole
    // entry gives inf: rows that may hold one multiply the lower pieces by
    // their finite values only
    const bool any_big = __builtin_amdgcn_ballot_w64(big) != 0;
#pragma unroll 1
    for (int mt = 0; mt < 4; ++mt) {
      // the small pieces' sums first: rounded at their own size, not at the result's
      f32x16 acc = {};
      if (__builtin_expect(!any_big, 1)) {
#pragma unroll
        for (int q = kPieces - 1; q >= 0; --q)
#pragma unroll
          for (int ks = 0; ks < 8; ++ks)
            acc = mfma<BF>(*reinterpret_cast<const u32x4*>(&rt[q][32 * mt + n][64 * h + 8 * ks]), x[ks], acc);
      } else {
#pragma unroll 1
        for (int q = kPieces - 1; q >= 0; --q) {
#pragma unroll
          for (int ks = 0; ks < 8; ++ks) {
            u32x4 xv = x[ks];
            __asm__ volatile("" : "+v"(xv));  // computed here, in this rare branch, not ahead of the loop
            acc = mfma<BF>(*reinterpret_cast<const u32x4*>(&rt[q][32 * mt + n][64 * h + 8 * ks]),
                           q == 0 ? xv : finite_only<BF>(xv), acc);
          }
        }
      }
      // lane (n, h): channels 32 mt + 16 h ..+ 15 of row n -> the wave's stage
      uint8_t* const st = &stage[wave][0];
      u32x4 o[2];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a = acc[2 * j] * unscale, b = acc[2 * j + 1] * unscale;
        o[j >> 2][j & 3] = BF ? pack_bf16(a, b) : static_cast<uint32_t>(f2h(a)) | (static_cast<uint32_t>(f2h(b)) << 16);
      }
      u32x4* dst = reinterpret_cast<u32x4*>(st + n * kStagePitch + 32 * h);
      dst[0] = o[0];
      dst[1] = o[1];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      // out in whole 64-byte row segments
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int rr = 16 * k + (lane >> 2);
        const u32x4 v = *reinterpret_cast<const u32x4*>(st + rr * kStagePitch + 16 * (lane & 3));
        if (r0 + rr < S)
          *reinterpret_cast<u32x4*>(out + (slice * S + r0 + rr) * kD + 32 * mt + 8 * (lane & 3)) = v;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
}

template <int BITS, bool BF, bool TOKEN>
void launch(const uint8_t* packed, const uint16_t* scale, int64_t BH, int64_t S, const float* R, uint16_t* out,
            hipStream_t st) {
  const int64_t slices = TOKEN ? 1 : BH, rows = TOKEN ? BH * S : S;
  const int cus = num_cus();
  const uint32_t blocks = static_cast<uint32_t>(cdiv(rows, kRows)), items = static_cast<uint32_t>(slices * blocks);
  const dim3 grid(items < static_cast<uint32_t>(cus) ? items : cus);
  hipLaunchKernelGGL((rotdq_kernel<BITS, BF, TOKEN>), grid, dim3(kThreads), 0, st, packed, scale, rows, blocks, items, R, out);
}

}  // namespace
}  // namespace fade

using namespace fade;

FADE_API int fade_rotate_dequant(const void* packed, const void* scale, int32_t dtype, int32_t bits, int32_t axis,
                                 int64_t B, int64_t H, int64_t S, int64_t D, const float* R, void* out, void* stream) {
  const char* fn = "fade_rotate_dequant";
  if (B < 0 || H < 0 || S < 0) return einval("%s: negative dimension", fn);
  if (D != kD) return einval("%s: head_dim must be %d, got %lld", fn, kD, (long long)D);
  if (bits != 2 && bits != 3 && bits != 4) return einval("%s: bits must be 2, 3 or 4, got %d", fn, bits);
  if (axis != FADE_AXIS_TOKEN && axis != FADE_AXIS_CHANNEL) return einval("%s: bad axis %d", fn, axis);
  if (dtype != FADE_DTYPE_F16 && dtype != FADE_DTYPE_BF16)
    return einval("%s: dtype must be FADE_DTYPE_F16 or FADE_DTYPE_BF16, got %d", fn, dtype);
  if (B * H * S == 0) return FADE_OK;
  if (B * H * S > (int64_t{1} << 35)) return einval("%s: shape too large", fn);  // work items are 32-bit
  if (packed == nullptr || scale == nullptr || R == nullptr || out == nullptr) return einval("%s: null pointer", fn);
  if (((reinterpret_cast<uintptr_t>(packed) | reinterpret_cast<uintptr_t>(R) | reinterpret_cast<uintptr_t>(out)) & 15) ||
      (reinterpret_cast<uintptr_t>(scale) & (axis == FADE_AXIS_CHANNEL ? 15 : 1)))
    return einval("%s: packed, R, out and a per-channel scale must be 16-byte aligned", fn);
  const uint8_t* pk = static_cast<const uint8_t*>(packed);
  const uint16_t* sc = static_cast<const uint16_t*>(scale);
  uint16_t* o = static_cast<uint16_t*>(out);
  hipStream_t st = as_stream(stream);
  const bool bf = dtype == FADE_DTYPE_BF16, token = axis == FADE_AXIS_TOKEN;
#define FADE_ROTDQ(BITS)                                                          \
  if (bf && token) launch<BITS, true, true>(pk, sc, B * H, S, R, o, st);          \
  else if (bf) launch<BITS, true, false>(pk, sc, B * H, S, R, o, st);             \
  else if (token) launch<BITS, false, true>(pk, sc, B * H, S, R, o, st);          \
  else launch<BITS, false, false>(pk, sc, B * H, S, R, o, st);
  if (bits == 4) { FADE_ROTDQ(4) }
  else if (bits == 2) { FADE_ROTDQ(2) }
  else { FADE_ROTDQ(3) }
#undef FADE_ROTDQ
  return check_launch(fn);
}
