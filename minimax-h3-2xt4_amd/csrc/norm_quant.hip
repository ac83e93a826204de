// DiT modulated RMSNorm, optionally fused with ConvRot256 and the per-row
// INT8 quantizer: the QKV / FC1 input preparation in one pass over x.
//
// One wavefront per row (a workgroup per row while the rows are few), lane l
// of a wavefront owning the 16-element units u = l + 64 j
// (elements [16u, 16u + 16)) as in the row quantizer, so loads and the int8
// store are 128-bit and contiguous across the wave. The sum of squares has a
// fixed order that does not depend on the launch: each lane adds its squares
// in (unit, element) order, then the 64 lane partials meet in an xor
// butterfly (offsets 32, 16, ..., 1); IEEE addition is commutative, so every
// lane ends with the same total. rsqrtf is replaced by a correctly rounded
// square root followed by a correctly rounded division.
#include "w8a8_device.h"
#include "w8a8_host.h"

#include <type_traits>

namespace w8a8 {

constexpr int kNormWaves = 4;

struct NormParams {
  const void* x;
  int64_t ldx, rows, cols;
  const float* weight;
  const float* shift;
  const float* mscale;
  int64_t ld_mod;
  int32_t mod_rows;
  float eps, inv_cols;
  const int32_t* labels;
  void* y;
  int64_t ldy;
  int8_t* q;
  int64_t ldq;
  float* qscale;
  const uint32_t* signs;   // ConvRot sign words (0 or 0x80000000 per column), or null
  bool shared;             // an output lies in x's memory (y == x: in place)
};

// MODE: 0 norm only, 1 quantize, 2 ConvRot256 (fp32) + quantize,
// 3 ConvRot256 rounded to the storage dtype + quantize; 2 or 3 | kNormSigned
// (4): the rotation takes the sign words (diag(s) then H), a compile-time
// choice so that the kernels without signs hold no registers for them.
constexpr int kNormSigned = 4;
template <int MODE>
constexpr int rot_of() { return (MODE & 3) == 2 ? 1 : (MODE & 3) == 3 ? 2 : 0; }

__device__ __forceinline__ void load16_f32(const float* p, float (&v)[16]) {
  const float4* q = reinterpret_cast<const float4*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 t = q[i];
    v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
  }
}

// Table flags of a kernel: kGain (weight present), kMod (shift/scale
// tables present), kAnyTables (decide per call from the pointers).
enum NormTables { kGain = 1, kMod = 2, kAnyTables = 4 };

// v: x on entry; on return the normalized, modulated value rounded to DT
// (as fp32; times 1/16 when SCALED), with its storage bits packed in bits.
template <int DT, int TB, bool SCALED>
__device__ __forceinline__ void modulate16(float (&v)[16], uint32_t (&bits)[8], float inv, const float* w,
                                           const float* sh, const float* sc, int64_t c0) {
  const bool gain = (TB & kGain) || ((TB & kAnyTables) && w);
  const bool mod = (TB & kMod) || ((TB & kAnyTables) && sh);
  float wv[16], shv[16], scv[16];
  if (gain) load16_f32(w + c0, wv);
  if (mod) {
    load16_f32(sc + c0, scv);
    load16_f32(sh + c0, shv);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    float t = DT == kF16 ? mul_mix(v[i], inv) : v[i] * inv;
    if (gain) t = t * wv[i];
    if (mod) {
      const float f = 1.0f + scv[i];
      t = t * f;
      t = t + shv[i];
    }
    v[i] = t;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if constexpr (DT == kF16) {
      bits[i] = f2h2_of_f32(v[2 * i], v[2 * i + 1]);
      v[2 * i] = h2f((uint16_t)(bits[i] & 0xffffu));
      v[2 * i + 1] = h2f((uint16_t)(bits[i] >> 16));
    } else {
      const uint16_t lo = f2bf(v[2 * i]), hi = f2bf(v[2 * i + 1]);
      bits[i] = (uint32_t)lo | ((uint32_t)hi << 16);
      v[2 * i] = bf2f(lo);
      v[2 * i + 1] = bf2f(hi);
    }
  }
  if constexpr (SCALED) scale16(v);
}

// Waves per workgroup of the norm-only kernel with AdaLN tables: the
// workgroup stages the gain and its first row's shift and scale rows in LDS,
// and its waves whose row carries that label read them there (the rows of a
// segment share the label). 16384 x 3072: 55 -> 41 us. With the rotation the
// tables' LDS costs more occupancy than the loads they save (61 -> 73 us).
constexpr int kNormStageWaves = 8;
constexpr int kNormStageMaxCols = 4096;   // 48 KB of tables

// Dynamic LDS of a W-wave workgroup: the rotation slots, then (STAGE) the
// gain, scale and shift rows.
template <int MODE, int W, bool STAGE>
constexpr int norm_lds_floats(int cols) { return (rot_of<MODE>() ? W * kRotWave : 0) + (STAGE ? 3 * cols : 0); }

// SPLIT: a workgroup of J waves takes one row. Every wave adds all the squares
// (the order is a chain through a lane's units), then normalizes, rotates and
// quantizes unit wave j alone; the maxima meet in LDS. For few rows, where a
// row per wave is one long chain of latencies on a part of the SIMDs; with
// more, the squares added J times over outweigh it. Row per wave / per
// workgroup, fp16 with AdaLN tables unless said: 353 x 5120 13.5 / 7.1 us, 353
// x 3072 8.9 / 5.9. Rows of up to four units a lane: 1536 x 3072 11.5 / 10.8,
// 1536 x 4096 14.6 / 12.5, 1536 x 3072 gain only 9.9 / 9.1, 1536 x 4096 bf16
// 18.5 / 16.2; 2048 x 3072 12.4 / 13.2, 2048 x 4096 bf16 19.7 / 20.9. Five and
// six units (a CU holds three such workgroups): 768 x 5376 16.9 / 12.4, 768 x
// 5120 bf16 18.4 / 18.5; 896 x 5376 16.4 / 17.9, 896 x 5120 bf16 18.1 / 23.6.
// Without the rounded rotation the chain is shorter (1536 x 4096 gain only,
// fp32 rotation: 10.8 / 11.5), and the smaller line serves.
constexpr int64_t split_rows(int jneed, int rot) { return jneed <= 4 && rot == 2 ? 1536 : 768; }

// WIDE: a rotated and rounded fp16 row waits for its scale as fp32, in the
// registers its x was widened into while the squares are added, not as fp16
// (KEEP16 below). Fewer conversions in a wave's chain, but more registers, so
// it is the faster one while its waves all fit the SIMDs at once (KEEP16 /
// WIDE, us): 2048 x 5376 21.5 / 21.1 and gain only 19.0 / 18.3, 2048 x 6144
// signed 26.2 / 24.4, 3072 x 5376 gain only 23.7 / 22.7, 3072 x 4096 21.0 /
// 20.6; past that 2560 x 5376 26.9 / 32.5, 4096 x 5376 gain only 27.9 / 31.4,
// 4096 x 4096 26.0 / 28.3. Rows of one or two units fit four waves to a SIMD
// either way and always take it (2048 x 2048 9.5 / 9.2, 8192 x 2048 23.5 /
// 23.2).
constexpr int64_t wide_rows(int j, int tables) { return j <= 2 ? INT64_MAX : j > 4 && (tables & kMod) ? 2048 : 3072; }

template <int DT, int MODE, int J, int TB, int W = kNormWaves, bool STAGE = false, bool SPLIT = false,
          bool WIDE = false>
__global__ __launch_bounds__(64 * W, J > 0 && J <= 6 && rot_of<MODE>() == 2 && DT == kF16 && !WIDE ? 4 : 1)
void norm_quant_kernel(NormParams p) {
  constexpr int ROT = rot_of<MODE>();
  constexpr bool PS = ROT != 0 && kPrescaled<DT>;
  // Rotated fp16 values wait for the row's scale as the fp16 they are rounded
  // to, eight registers a unit instead of sixteen; the maximum is taken on the
  // fp32 rotation and rounded once (rounding is monotonic and odd). With x
  // held in its storage type too, six units take 128 registers instead of 178:
  // four waves per SIMD instead of two (6814 x 5376 63 -> 48 us; with the sign
  // words four registers spill there, 6144 x 6144 66 -> 61 us all the same).
  constexpr bool KEEP16 = J > 0 && ROT == 2 && DT == kF16 && !WIDE;
  static_assert(!WIDE || (J > 0 && ROT == 2 && DT == kF16 && !SPLIT), "the other storage of KEEP16's rows");
  static_assert(!SPLIT || (W == J && !STAGE && MODE != 0), "one unit per wave");
  __shared__ float wmax[SPLIT ? W : 1];
  static_assert(!STAGE || (TB == (kGain | kMod) && ROT == 0), "staged tables: norm-only DiT form");
  extern __shared__ __attribute__((aligned(16))) float dsm[];
  float* const lds = dsm;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t row0 = SPLIT ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * W;
  const int64_t row = SPLIT ? row0 : row0 + wave;
  float* const tw = dsm + (ROT ? W * kRotWave : 0);
  float* const tsc = tw + p.cols;
  float* const tsh = tsc + p.cols;
  int l0 = -1;
  if constexpr (STAGE) {
    // Every thread reaches the barrier before any row bound is applied.
    l0 = min(max(p.labels[row0], 0), p.mod_rows - 1);
    const float4* gw = reinterpret_cast<const float4*>(p.weight);
    const float4* gsc = reinterpret_cast<const float4*>(p.mscale + (int64_t)l0 * p.ld_mod);
    const float4* gsh = reinterpret_cast<const float4*>(p.shift + (int64_t)l0 * p.ld_mod);
    const int n4 = (int)(p.cols >> 2);
    for (int i = threadIdx.x; i < n4; i += 64 * W) {
      reinterpret_cast<float4*>(tw)[i] = gw[i];
      reinterpret_cast<float4*>(tsc)[i] = gsc[i];
      reinterpret_cast<float4*>(tsh)[i] = gsh[i];
    }
    __syncthreads();
  }
  if (row >= p.rows) return;
  const int units = (int)(p.cols >> 4);
  const int jcount = (units + 63) >> 6;
  const uint16_t* xrow = reinterpret_cast<const uint16_t*>(p.x) + row * p.ldx;
  uint16_t* yrow = p.y ? reinterpret_cast<uint16_t*>(p.y) + row * p.ldy : nullptr;
  const float* sh = nullptr;
  const float* sc = nullptr;
  bool staged = false;
  if ((TB & kMod) || ((TB & kAnyTables) && p.shift)) {
    const int l = min(max(p.labels[row], 0), p.mod_rows - 1);
    staged = STAGE && l == l0;
    sh = p.shift + (int64_t)l * p.ld_mod;
    sc = p.mscale + (int64_t)l * p.ld_mod;
  }
  float* buf = ROT ? rot_slot(lds, wave, lane) : nullptr;
  const int t = lane & 15;

  // Normalize one unit (v holds x), store y, rotate for the quantizer.
  auto finish = [&](int u, float (&v)[16], float inv, bool store_y) {
    uint32_t bits[8];
    if (STAGE && staged) modulate16<DT, TB, PS>(v, bits, inv, tw, tsh, tsc, (int64_t)u * 16);
    else modulate16<DT, TB, PS>(v, bits, inv, p.weight, sh, sc, (int64_t)u * 16);
    if (store_y && yrow) {
      uint4* dst = reinterpret_cast<uint4*>(yrow + (int64_t)u * 16);
      dst[0] = make_uint4(bits[0], bits[1], bits[2], bits[3]);
      dst[1] = make_uint4(bits[4], bits[5], bits[6], bits[7]);
    }
    if constexpr (ROT != 0) {
      constexpr bool SG = (MODE & kNormSigned) != 0;
      convrot256_lanes<true, SG, PS>(v, buf, t, SG ? p.signs + 256 * (u >> 4) : nullptr);
      if constexpr (ROT == 2 && !KEEP16) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = round_to<DT>(v[i]);
      }
    }
  };
  auto store_q = [&](int u, const float (&v)[16], float s, float rcp) {
    *reinterpret_cast<uint4*>(p.q + row * p.ldq + (int64_t)u * 16) =
        ROT == 1 && (SPLIT || J != 2) ? quant16(v, s, rcp) : quant16_each(v, s, rcp);
  };
  // ss + x*x with one rounding: the square of a 16-bit float is exact in
  // fp32 (at most 22 significant bits, no overflow or underflow), so the FMA
  // equals the separately rounded product and sum.
  auto add_squares = [](float ss, const float (&v)[16]) {
#pragma unroll
    for (int i = 0; i < 16; ++i) ss = __builtin_fmaf(v[i], v[i], ss);
    return ss;
  };
  auto inv_rms = [&](float ss) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) ss = ss + __shfl_xor(ss, off, 64);
    const float mean = ss * p.inv_cols;
    const float d = mean + p.eps;
    return 1.0f / __builtin_sqrtf(d);
  };

  if constexpr (J > 0) {
    // The row waits in its storage type between the two passes over it (bf16
    // rows of up to four units a lane widened, in the registers of their
    // results: 16384 x 3072 64.5 us, 73.2 widened twice; six units unrotated
    // too, with 166 registers instead of 174 that is three waves to a SIMD and
    // not two: 16384 x 5376 112 / 128 us).
    constexpr bool HOLD32 = WIDE || (DT == kBF16 && MODE != 0 && (J <= 4 || MODE == 1));
    uint4 raw[J][4];
    float keep[MODE != 0 && !KEEP16 ? J : 1][16];
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < J; ++j)
      if (!WIDE && lane + 64 * j < units) raw16<DT>(xrow + (int64_t)(lane + 64 * j) * 16, raw[j]);
    // (WIDE: loads beside the adds, so that the first units' squares need not
    // wait for the last: 2048 x 5376 gain only 18.9 -> 18.3 us.)
#pragma unroll
    for (int j = 0; j < J; ++j) {
      if (lane + 64 * j < units) {
        if constexpr (WIDE) raw16<DT>(xrow + (int64_t)(lane + 64 * j) * 16, raw[j]);
        float tmp[16];
        float (&v)[16] = HOLD32 ? keep[HOLD32 ? j : 0] : tmp;
        unpack16<DT>(raw[j], v);
        ss = add_squares(ss, v);
      }
    }
    const float inv = inv_rms(ss);
    float amax = 0.0f;
    uint32_t h16[KEEP16 ? J : 1][8];
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int u = lane + 64 * j;
      if ((!SPLIT || j == wave) && u < units) {
        float (&v)[16] = keep[MODE != 0 && !KEEP16 ? j : 0];
        if constexpr (!HOLD32) unpack16<DT>(raw[j], v);
        finish(u, v, inv, true);
        if constexpr (MODE != 0) {
#pragma unroll
          for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(v[i]));
        }
        if constexpr (KEEP16) {
#pragma unroll
          for (int i = 0; i < 8; ++i) h16[j][i] = f2h2_of_f32(v[2 * i], v[2 * i + 1]);
        }
      }
    }
    if constexpr (MODE != 0) {
      amax = wave_max(amax);
      if constexpr (SPLIT) {
        if (lane == 0) wmax[wave] = amax;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < J; ++j) amax = fmaxf(amax, wmax[j]);
      }
      if constexpr (KEEP16) amax = round_to<DT>(amax);
      const float s = row_scale_of(amax);
      const float rcp = 1.0f / s;
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int u = lane + 64 * j;
        if ((!SPLIT || j == wave) && u < units) {
          if constexpr (KEEP16) {
            float v[16];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              v[2 * i] = h2f((uint16_t)(h16[j][i] & 0xffffu));
              v[2 * i + 1] = h2f((uint16_t)(h16[j][i] >> 16));
            }
            store_q(u, v, s, rcp);
          } else {
            store_q(u, keep[j], s, rcp);
          }
        }
      }
      if (lane == 0 && (!SPLIT || wave == 0)) p.qscale[row] = s;
    }
  } else {
    // Rows too wide for registers: sum of squares, then absmax, then the
    // stores, each pass re-reading x.
    float ss = 0.0f;
    for (int j = 0; j < jcount; ++j) {
      const int u = lane + 64 * j;
      if (u < units) {
        float v[16];
        load16<DT>(xrow + (int64_t)u * 16, v);
        ss = add_squares(ss, v);
      }
    }
    const float inv = inv_rms(ss);
    float s = 0.0f, rcp = 0.0f;
    if constexpr (MODE != 0) {
      float amax = 0.0f;
      for (int j = 0; j < jcount; ++j) {
        const int u = lane + 64 * j;
        if (u < units) {
          float v[16];
          load16<DT>(xrow + (int64_t)u * 16, v);
          finish(u, v, inv, false);
#pragma unroll
          for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(v[i]));
        }
      }
      amax = wave_max(amax);
      s = row_scale_of(amax);
      rcp = 1.0f / s;
    }
    for (int j = 0; j < jcount; ++j) {
      const int u = lane + 64 * j;
      if (u < units) {
        float v[16];
        load16<DT>(xrow + (int64_t)u * 16, v);
        finish(u, v, inv, true);
        if constexpr (MODE != 0) store_q(u, v, s, rcp);
      }
    }
    if constexpr (MODE != 0) {
      if (lane == 0) p.qscale[row] = s;
    }
  }
}

template <int DT, int MODE, int TB, int W = kNormWaves, bool STAGE = false>
static void launch_norm_j(const NormParams& p, hipStream_t stream) {
  const int jneed = (int)(((p.cols >> 4) + 63) / 64);
  const dim3 grid((unsigned)((p.rows + W - 1) / W)), block(64 * W);
  const size_t lds = 4 * (size_t)max(norm_lds_floats<MODE, W, STAGE>((int)p.cols), 1);
  if constexpr (MODE != 0 && !STAGE) {
    // A row per workgroup while the rows are few; not in place, where a wave
    // would store its unit while another still reads the row.
    if (jneed >= 2 && jneed <= 6 && p.rows <= split_rows(jneed, rot_of<MODE>()) && !p.shared) {
      const dim3 rows((unsigned)p.rows);
      auto go = [&](auto j_tag) {
        constexpr int JJ = decltype(j_tag)::value;
        hipLaunchKernelGGL((norm_quant_kernel<DT, MODE, JJ, TB, JJ, false, true>), rows, dim3(64 * JJ),
                           4 * (size_t)max(norm_lds_floats<MODE, JJ, false>(0), 1), stream, p);
      };
      switch (jneed) {
        case 2: go(std::integral_constant<int, 2>{}); break;
        case 3: go(std::integral_constant<int, 3>{}); break;
        case 4: go(std::integral_constant<int, 4>{}); break;
        case 5: go(std::integral_constant<int, 5>{}); break;
        default: go(std::integral_constant<int, 6>{}); break;
      }
      return;
    }
  }
  auto go = [&](auto j_tag) {
    constexpr int JJ = decltype(j_tag)::value;
    if constexpr (DT == kF16 && rot_of<MODE>() == 2 && JJ > 0 && JJ <= 6) {
      if (p.rows <= wide_rows(JJ, TB)) {
        hipLaunchKernelGGL((norm_quant_kernel<DT, MODE, JJ, TB, W, STAGE, false, true>), grid, block, lds, stream, p);
        return;
      }
    }
    if constexpr (!(DT == kF16 && rot_of<MODE>() == 2) || JJ == 0 || JJ > 2)
      hipLaunchKernelGGL((norm_quant_kernel<DT, MODE, JJ, TB, W, STAGE>), grid, block, lds, stream, p);
  };
  switch (jneed) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: case 6: go(std::integral_constant<int, 6>{}); break;
    case 7: case 8: go(std::integral_constant<int, 8>{}); break;
    default: go(std::integral_constant<int, 0>{}); break;
  }
}

// Rows held in registers for the DiT (gain + AdaLN tables) and plain
// RMSNorm (gain only) forms; other table combinations take the streaming
// kernel with the tables decided per call.
template <int DT, int MODE>
static int launch_norm(const NormParams& p, hipStream_t stream) {
  if (MODE == 0 && p.weight && p.shift && p.cols <= kNormStageMaxCols) {
    if constexpr (MODE == 0) launch_norm_j<DT, MODE, kGain | kMod, kNormStageWaves, true>(p, stream);
  } else if (p.weight && p.shift) {
    launch_norm_j<DT, MODE, kGain | kMod>(p, stream);
  } else if (p.weight) {
    launch_norm_j<DT, MODE, kGain>(p, stream);
  } else {
    const dim3 grid((unsigned)((p.rows + kNormWaves - 1) / kNormWaves)), block(64 * kNormWaves);
    hipLaunchKernelGGL((norm_quant_kernel<DT, MODE, 0, kAnyTables>), grid, block,
                       4 * (size_t)max(norm_lds_floats<MODE, kNormWaves, false>(0), 1), stream, p);
  }
  return launch_status("w8a8_norm_quantize");
}

// Whether [a, a + an) and [b, b + bn) share a byte.
static bool spans_overlap(const void* a, int64_t an, const void* b, int64_t bn) {
  const uintptr_t pa = (uintptr_t)a, pb = (uintptr_t)b;
  return pa < pb + (uintptr_t)bn && pb < pa + (uintptr_t)an;
}

}  // namespace w8a8

extern "C" int w8a8_norm_quantize(const W8A8NormArgs* a) {
  using namespace w8a8;
  W8A8_REQUIRE(a != nullptr, "w8a8_norm_quantize: null args");
  W8A8_REQUIRE(a->struct_size == sizeof(W8A8NormArgs), "w8a8_norm_quantize: struct_size %u != %zu",
               a->struct_size, sizeof(W8A8NormArgs));
  W8A8_REQUIRE(a->x_dtype == W8A8_F16 || a->x_dtype == W8A8_BF16, "w8a8_norm_quantize: x_dtype %d not F16/BF16",
               a->x_dtype);
  W8A8_REQUIRE(a->rows >= 0 && a->cols >= 0, "w8a8_norm_quantize: negative shape");
  W8A8_REQUIRE(a->y != nullptr || a->q != nullptr, "w8a8_norm_quantize: neither y nor q requested");
  W8A8_REQUIRE(a->convrot == 0 || a->convrot == 256, "w8a8_norm_quantize: convrot must be 0 or 256");
  W8A8_REQUIRE(a->round_rotated == 0 || a->round_rotated == 1, "w8a8_norm_quantize: round_rotated must be 0 or 1");
  const int group = (a->q && a->convrot) ? 256 : 16;
  W8A8_REQUIRE(a->cols % group == 0, "w8a8_norm_quantize: cols %lld not a multiple of %d", (long long)a->cols,
               group);
  W8A8_REQUIRE(a->cols <= ((int64_t)1 << 30), "w8a8_norm_quantize: cols too large");
  W8A8_REQUIRE((a->mod_shift == nullptr) == (a->mod_scale == nullptr),
               "w8a8_norm_quantize: mod_shift and mod_scale go together");
  if (a->rows == 0) return W8A8_OK;
  W8A8_REQUIRE(a->cols > 0, "w8a8_norm_quantize: zero-width rows have no norm");
  W8A8_REQUIRE(a->x != nullptr && aligned16(a->x) && a->ldx >= a->cols && (a->ldx * 2) % 16 == 0,
               "w8a8_norm_quantize: x must be 16-byte aligned with ldx >= cols and a 16-byte row stride");
  if (a->y) {
    W8A8_REQUIRE(aligned16(a->y) && a->ldy >= a->cols && (a->ldy * 2) % 16 == 0,
                 "w8a8_norm_quantize: y must be 16-byte aligned with ldy >= cols and a 16-byte row stride");
  }
  if (a->q) {
    W8A8_REQUIRE(a->q_scale != nullptr, "w8a8_norm_quantize: q requires q_scale");
    W8A8_REQUIRE(aligned16(a->q) && a->ldq >= a->cols && a->ldq % 16 == 0,
                 "w8a8_norm_quantize: q must be 16-byte aligned with ldq >= cols, a multiple of 16");
  }
  W8A8_REQUIRE(a->weight == nullptr || aligned16(a->weight), "w8a8_norm_quantize: weight must be 16-byte aligned");
  if (a->mod_shift) {
    W8A8_REQUIRE(a->labels != nullptr && a->mod_rows >= 1, "w8a8_norm_quantize: modulation needs labels, mod_rows");
    W8A8_REQUIRE(aligned16(a->mod_shift) && aligned16(a->mod_scale) && a->ld_mod >= a->cols && a->ld_mod % 4 == 0,
                 "w8a8_norm_quantize: tables must be 16-byte aligned with ld_mod >= cols, a multiple of 4");
  }
  NormParams p;
  p.x = a->x;
  p.ldx = a->ldx;
  p.rows = a->rows;
  p.cols = a->cols;
  p.weight = a->weight;
  p.shift = a->mod_shift;
  p.mscale = a->mod_scale;
  p.ld_mod = a->ld_mod;
  p.mod_rows = a->mod_rows;
  p.eps = a->eps;
  // fp32(1/cols), the constant the reference multiplies the sum by.
  p.inv_cols = (float)(1.0 / (double)a->cols);
  p.labels = a->labels;
  p.y = a->y;
  p.ldy = a->ldy;
  p.q = a->q;
  p.ldq = a->ldq;
  p.qscale = a->q_scale;
  const int64_t xbytes = ((a->rows - 1) * a->ldx + a->cols) * 2;
  p.shared = (a->y && spans_overlap(a->x, xbytes, a->y, ((a->rows - 1) * a->ldy + a->cols) * 2)) ||
             (a->q && (spans_overlap(a->x, xbytes, a->q, (a->rows - 1) * a->ldq + a->cols) ||
                       spans_overlap(a->x, xbytes, a->q_scale, a->rows * 4)));
  W8A8_REQUIRE(a->convrot_signs == nullptr || (a->q && a->convrot && aligned16(a->convrot_signs)),
               "w8a8_norm_quantize: convrot_signs needs q, convrot and a 16-byte aligned array");
  p.signs = a->convrot_signs;
  hipStream_t stream = reinterpret_cast<hipStream_t>(a->stream);
  const int mode = (a->q == nullptr ? 0 : a->convrot == 0 ? 1 : a->round_rotated ? 3 : 2) |
                   (a->convrot_signs ? kNormSigned : 0);
  if (a->x_dtype == W8A8_F16) {
    switch (mode) {
      case 0: return launch_norm<kF16, 0>(p, stream);
      case 1: return launch_norm<kF16, 1>(p, stream);
      case 2: return launch_norm<kF16, 2>(p, stream);
      case 3: return launch_norm<kF16, 3>(p, stream);
      case 6: return launch_norm<kF16, 6>(p, stream);
      default: return launch_norm<kF16, 7>(p, stream);
    }
  }
  switch (mode) {
    case 0: return launch_norm<kBF16, 0>(p, stream);
    case 1: return launch_norm<kBF16, 1>(p, stream);
    case 2: return launch_norm<kBF16, 2>(p, stream);
    case 3: return launch_norm<kBF16, 3>(p, stream);
    case 6: return launch_norm<kBF16, 6>(p, stream);
    default: return launch_norm<kBF16, 7>(p, stream);
  }
}
