// Expert products of a small forward batch (decode steps, short prompts): few
// routed rows per expert, so the whole cost is streaming the touched experts'
// weights once.
//
// Reference: abacus/moe/moe.py:78-80 (x w_gate, x w_up, (silu(gate) up) w_down
// per expert), as the grouped GEMMs of grouped_gemm.hip; rows are the same
// expert-contiguous rows.
#include <algorithm>

#include "common.h"

namespace abacus {
namespace {

typedef __bf16 dec_bf16x8 __attribute__((ext_vector_type(8)));
typedef float dec_f32x4 __attribute__((ext_vector_type(4)));

constexpr int kGroup = 16;       // rows per MFMA
constexpr int kRows = 2 * kGroup;  // rows per pass over a tile's weights
constexpr int kKB = 32;     // k rows per wave step: 8 for each of the 4 lane groups

// A wave's step takes 32 k rows x 16 lanes x 16 bytes of a weight matrix
// (128 bf16 or 64 fp32 columns): lane l loads the 16 bytes of its columns
// 16-byte group l % 16 in the 8 rows 8 (l / 16) .. +7, straight to registers.
template <typename T> constexpr int kVec = 16 / (int)sizeof(T);
template <typename T> constexpr int kCols = 16 * kVec<T>;

// Weight rows of a hidden size that is not whole vectors start at any element;
// the hardware takes vector loads at any address, so only the type says so.
// NT: nontemporal, for weights that a call reads once and the caches cannot hold.
template <typename T, bool UNALIGNED, bool NT>
__device__ inline Vec16 load_weights(const T* p) {
  if constexpr (UNALIGNED) {
    typedef uint32_t u32x4_ua __attribute__((ext_vector_type(4), aligned(2)));
    const u32x4_ua* q = reinterpret_cast<const u32x4_ua*>(p);
    const u32x4_ua v = NT ? __builtin_nontemporal_load(q) : *q;
    Vec16 r;
    r.w[0] = v.x; r.w[1] = v.y; r.w[2] = v.z; r.w[3] = v.w;
    return r;
  } else {
    return NT ? ld16_stream(p) : ld16(p);
  }
}

// acc[j] += x rows (16) x the step's columns: column j of every lane's vector
// is one MFMA, whose operand element k is row 8 (l / 16) + i of lane l's loads.
__device__ inline void step_mfma(dec_f32x4 (&acc)[8], const Vec16 (&w)[8], const Vec16 (&x)[1]) {
  const dec_bf16x8 a = __builtin_bit_cast(dec_bf16x8, x[0]);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    Vec16 b;  // rows 0..7 of column j: an 8 x 8 transpose in registers, one v_perm per dword
#pragma unroll
    for (int p = 0; p < 4; ++p)
      b.w[p] = __builtin_amdgcn_perm(w[2 * p + 1].w[j >> 1], w[2 * p].w[j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
    acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(dec_bf16x8, b), acc[j], 0, 0, 0);
  }
}
__device__ inline void step_mfma(dec_f32x4 (&acc)[4], const Vec16 (&w)[8], const Vec16 (&x)[2]) {
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bits_f32(x[i >> 2].w[i & 3]), bits_f32(w[i].w[j]), acc[j], 0, 0, 0);
}

// One step's operands: the weight vectors and, per 16-row group, the 8
// consecutive k of this lane's row.
constexpr int RG = kRows / kGroup;
template <typename T>
struct Step {
  static constexpr int XV = 8 / kVec<T>;
  Vec16 w[8];
  Vec16 x[RG][XV];
};

// acc += x[rows] * w over the k-blocks kb0, kb0 + kstride, ... < kb1 (32 rows
// each) of a reduction of K rows.  w: the matrix's first row at the tile's
// first column; x: the first of n_rows rows (16 per group are taken, those past
// the last one repeating it), pitch elements apart and zero from K to the next
// whole vector.  Everything but w, x and the lane is wave-uniform, so a load is
// a scalar base plus one of two lane offsets.
template <typename T, bool UNALIGNED, bool NT>
__device__ inline void stream_rows(const T* __restrict__ w, int64_t ldw, const T* __restrict__ x, int64_t pitch,
                                   int n_rows, int K, int kb0, int kb1, int kstride, int lane,
                                   dec_f32x4 (&acc)[RG][kVec<T>]) {
  using S = Step<T>;
  const int kl = 8 * (lane >> 4);
  const uint32_t woff = (uint32_t)kl * (uint32_t)ldw + kVec<T> * (lane & 15);
  uint32_t xoff[RG];
#pragma unroll
  for (int r = 0; r < RG; ++r) xoff[r] = (uint32_t)min(r * kGroup + (lane & 15), n_rows - 1) * (uint32_t)pitch + kl;
  auto load = [&](S& s, int kb) __attribute__((always_inline)) {
    const T* wb = w + (int64_t)kb * kKB * ldw;
    const T* xb = x + (int64_t)kb * kKB;
#pragma unroll
    for (int i = 0; i < 8; ++i) s.w[i] = load_weights<T, UNALIGNED, NT>(wb + i * ldw + woff);
#pragma unroll
    for (int r = 0; r < RG; ++r)
      if (r * kGroup < n_rows) {
#pragma unroll
        for (int v = 0; v < S::XV; ++v) s.x[r][v] = ld16(xb + v * kVec<T> + xoff[r]);
      }
  };
  auto use = [&](const S& s) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < RG; ++r)
      if (r * kGroup < n_rows) step_mfma(acc[r], s.w, s.x[r]);
  };
  const int whole = min(kb1, K / kKB);  // k-blocks without a tail
  S a, b;
  int kb = kb0;
  if (kb < whole) load(a, kb);
  while (kb < whole) {  // the next block's loads go out before this one's products
    if (kb + kstride < whole) load(b, kb + kstride);
    use(a);
    kb += kstride;
    if (kb >= whole) break;
    if (kb + kstride < whole) load(a, kb + kstride);
    use(b);
    kb += kstride;
  }
  if (kb < kb1) {  // this wave's is the tail block: rows from K on read row K - 1 and count as zero
    const int k = kb * kKB + kl;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      a.w[i] = load_weights<T, UNALIGNED, NT>(w + (int64_t)min(k + i, K - 1) * ldw + kVec<T> * (lane & 15));
      if (k + i >= K) a.w[i] = zero16();
    }
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int v = 0; v < S::XV; ++v) {
        const bool in = k + v * kVec<T> < K;
        a.x[r][v] = in ? ld16(x + (int64_t)kb * kKB + v * kVec<T> + xoff[r]) : zero16();
      }
    use(a);
  }
}

// This lane's part of a wave's 16 x kCols partial product, row-major in LDS:
// rows 4 (l / 16) + q, columns kVec (l % 16) .. +kVec-1.
template <typename T>
__device__ inline void store_partial(float* part, const dec_f32x4 (&acc)[kVec<T>], int lane) {
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int j = 0; j < kVec<T>; j += 4)
      *reinterpret_cast<float4*>(part + (4 * (lane >> 4) + q) * kCols<T> + kVec<T> * (lane & 15) + j) =
          make_float4(acc[j][q], acc[j + 1][q], acc[j + 2][q], acc[j + 3][q]);
}

template <typename T>
__device__ inline void store4(T* p, float a, float b, float c, float d) {
  if constexpr (sizeof(T) == 2) {
    typedef uint32_t u32x2_ua __attribute__((ext_vector_type(2), aligned(2)));
    u32x2_ua v;
    v.x = pack_bf16x2(a, b);
    v.y = pack_bf16x2(c, d);
    *reinterpret_cast<u32x2_ua*>(p) = v;
  } else {
    typedef float f32x4_ua __attribute__((ext_vector_type(4), aligned(4)));
    *reinterpret_cast<f32x4_ua*>(p) = f32x4_ua{a, b, c, d};
  }
}

// What bounds these kernels is the weight stream, so the weights go from HBM to
// registers to MFMA with no LDS and no barrier on the way, each wave keeping 8 KB
// of loads in flight under its products, and a tile's reduction is split over
// the block's waves.  A block of 4 waves leaves a CU room for a second one, whose
// loads cover the first one's start and sums; where the tiles are fewer than two
// per CU, 8 waves split each further.  Measured (us, both products, against the
// 256-column tiles of grouped_gemm.hip): bf16 E 8 D 4096 M 14336, 1 token top-2
// 242 -> 120 (5.9 TB/s; 4 waves 155), 64 tokens 569 -> 487; E 64 D 2048 M 1408,
// 64 tokens top-6 220 -> 179, 128 tokens 225 -> 186; fp32 E 16 D 1024 M 2816, 1
// token 352 -> 31, 128 tokens 493 -> 136.  Nontemporal weight loads 8% of it; a
// third step in flight spills (+15%); 64 rows a pass spills too.

// H = silu(x w_gate) (x w_up) for one expert's rows and kCols columns per
// block.  The first half of the W waves share w_gate's k-blocks, the second
// half w_up's; the partial products meet in LDS and are added in wave order.
template <typename T, int W, bool UNALIGNED, bool NT>
__global__ __launch_bounds__(W * 64, 2) void decode_gateup_kernel(const T* __restrict__ xp,
                                                                    const T* __restrict__ w_gate,
                                                                    const T* __restrict__ w_up,
                                                                    const int32_t* __restrict__ offsets, int D, int M,
                                                                    int64_t ldh, T* __restrict__ h) {
  constexpr int HW = W / 2;  // waves per matrix
  constexpr int NC = kCols<T>, PART = kGroup * NC;
  __shared__ __attribute__((aligned(16))) float part[W * PART];
  const int e = blockIdx.y;
  const int row0 = offsets[e], row1 = offsets[e + 1];
  if (row0 == row1) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave / HW;
  const int n0 = min((int)blockIdx.x * NC, M - NC);  // the last tile overlaps its neighbour: the same sums, written twice
  const T* w = (half ? w_up : w_gate) + (int64_t)e * D * M + n0;
  for (int r0 = row0 + (int)blockIdx.z * kRows; r0 < row1; r0 += (int)gridDim.z * kRows) {
    dec_f32x4 acc[RG][kVec<T>] = {};
    stream_rows<T, UNALIGNED, NT>(w, M, xp + (int64_t)r0 * D, D, row1 - r0, D, wave % HW, (D + kKB - 1) / kKB, HW, lane,
                                  acc);
#pragma unroll
    for (int r = 0; r < RG; ++r) {
      const int rg0 = r0 + r * kGroup;
      if (rg0 >= row1) break;
      __syncthreads();  // the previous group's sums are read
      store_partial<T>(part + wave * PART, acc[r], lane);
      __syncthreads();
      for (int v = tid; v < PART / 4; v += W * 64) {
        const int row = rg0 + v / (NC / 4), c = (v % (NC / 4)) * 4;
        if (row >= row1) continue;
        float s[2][4];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          float4 t = *reinterpret_cast<const float4*>(part + HW * hf * PART + 4 * v);
#pragma unroll
          for (int p = 1; p < HW; ++p) {
            const float4 u = *reinterpret_cast<const float4*>(part + (HW * hf + p) * PART + 4 * v);
            t.x += u.x; t.y += u.y; t.z += u.z; t.w += u.w;
          }
          s[hf][0] = t.x; s[hf][1] = t.y; s[hf][2] = t.z; s[hf][3] = t.w;
        }
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // each product rounded to the dtype, as the separate products are
          const float g = round_to<T>(s[0][i]), u = round_to<T>(s[1][i]);
          o[i] = round_to<T>(silu_f32(g)) * u;
        }
        store4<T>(h + (int64_t)row * ldh + n0 + c, o[0], o[1], o[2], o[3]);
      }
      if (blockIdx.x == gridDim.x - 1 && tid < kGroup && rg0 + tid < row1)  // H's pad columns
        for (int64_t c = M; c < ldh; ++c) h[(int64_t)(rg0 + tid) * ldh + c] = (T)0;
    }
  }
}

// Y = H w_down for one expert's rows, kCols columns and one slice of the
// k-blocks per block, shared by its W waves.  One slice: Y itself; more: fp32
// partials [slice][R][D] for decode_reduce_kernel.
template <typename T, int W, bool NT>
__global__ __launch_bounds__(W * 64, 2) void decode_down_kernel(const T* __restrict__ h, const T* __restrict__ w_down,
                                                                  const int32_t* __restrict__ offsets, int M, int D,
                                                                  int64_t ldh, int64_t R, int kb_per, int slices,
                                                                  T* __restrict__ y, float* __restrict__ ws) {
  constexpr int NC = kCols<T>, PART = kGroup * NC;
  __shared__ __attribute__((aligned(16))) float part[W * PART];
  const int e = blockIdx.y;
  const int row0 = offsets[e], row1 = offsets[e + 1];
  if (row0 == row1) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = min((int)blockIdx.x * NC, D - NC);
  const int nkb = (M + kKB - 1) / kKB, slice = (int)blockIdx.z % slices, kb0 = slice * kb_per, kb1 = min(kb0 + kb_per, nkb);
  const T* w = w_down + (int64_t)e * M * D + n0;
  const int chunk = (int)blockIdx.z / slices, chunks = (int)gridDim.z / slices;
  for (int r0 = row0 + chunk * kRows; r0 < row1; r0 += chunks * kRows) {
    dec_f32x4 acc[RG][kVec<T>] = {};
    stream_rows<T, false, NT>(w, D, h + (int64_t)r0 * ldh, ldh, row1 - r0, M, kb0 + wave, kb1, W, lane, acc);
#pragma unroll
    for (int r = 0; r < RG; ++r) {
      const int rg0 = r0 + r * kGroup;
      if (rg0 >= row1) break;
      __syncthreads();
      store_partial<T>(part + wave * PART, acc[r], lane);
      __syncthreads();
      for (int v = tid; v < PART / 4; v += W * 64) {
        const int row = rg0 + v / (NC / 4), c = (v % (NC / 4)) * 4;
        if (row >= row1) continue;
        float4 t = *reinterpret_cast<const float4*>(part + 4 * v);
#pragma unroll
        for (int p = 1; p < W; ++p) {
          const float4 u = *reinterpret_cast<const float4*>(part + p * PART + 4 * v);
          t.x += u.x; t.y += u.y; t.z += u.z; t.w += u.w;
        }
        if (slices == 1) store4<T>(y + (int64_t)row * D + n0 + c, t.x, t.y, t.z, t.w);
        else *reinterpret_cast<float4*>(ws + ((int64_t)slice * R + row) * D + n0 + c) = t;
      }
    }
  }
}

// Y = the slices' partials added in slice order, four elements a thread.
template <typename T>
__global__ __launch_bounds__(256) void decode_reduce_kernel(const float* __restrict__ ws, int64_t n, int slices,
                                                            T* __restrict__ y) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  float4 t = *reinterpret_cast<const float4*>(ws + i);
  for (int s = 1; s < slices; ++s) {
    const float4 u = *reinterpret_cast<const float4*>(ws + s * n + i);
    t.x += u.x; t.y += u.y; t.z += u.z; t.w += u.w;
  }
  store4<T>(y + i, t.x, t.y, t.z, t.w);
}

// Blocks of 4 waves from about two tiles per CU on, of 8 below (see above).
bool four_waves(int64_t tiles) { return tiles >= 512; }

// k-blocks per slice of the down projection: enough slices for about two
// blocks on each of 256 CUs, at least two k-blocks per wave.
struct DownPlan {
  int kb_per, slices;
};
DownPlan plan_down(int64_t R, int64_t D, int64_t M, int64_t E, int cols) {
  const int64_t tiles = (D + cols - 1) / cols * std::min(E, R);
  const int64_t nkb = (M + kKB - 1) / kKB;
  const int64_t s = std::max<int64_t>(1, std::min<int64_t>(512 / tiles, nkb / 16));
  const int64_t per = (nkb + s - 1) / s;
  return {(int)per, (int)((nkb + per - 1) / per)};
}

template <typename T, int W, bool UNALIGNED, bool NT>
void launch_gateup(dim3 grid, hipStream_t s, const void* xp, const void* wg, const void* wu, const int32_t* offsets,
                   int64_t D, int64_t M, int64_t ldh, void* h) {
  hipLaunchKernelGGL((decode_gateup_kernel<T, W, UNALIGNED, NT>), grid, dim3(W * 64), 0, s, (const T*)xp, (const T*)wg,
                     (const T*)wu, offsets, (int)D, (int)M, ldh, (T*)h);
}

template <typename T, bool NT>
int launch(const void* xp, const void* wg, const void* wu, const void* wd, const int32_t* offsets, int64_t R, int64_t D,
           int64_t M, int64_t E, int64_t ldh, void* h, void* y, float* ws, hipStream_t s) {
  constexpr int NC = kCols<T>;
  // An expert's passes of 32 rows run beside each other, up to four: one expert
  // may hold many of the rows (E 4 D 512 M 1024, 128 tokens top-1: 26 -> 19 us).
  // They are the slowest grid dimension, so that the blocks without rows come
  // last: between the others they left CUs idle (E 64, 64 tokens: 179 -> 484 us).
  const unsigned chunks = (unsigned)std::min<int64_t>(4, (R + kRows - 1) / kRows);
  const unsigned t1 = (unsigned)((M + NC - 1) / NC), t2 = (unsigned)((D + NC - 1) / NC);
  const DownPlan p = plan_down(R, D, M, E, NC);
  const int64_t touched = std::min(E, R);
  const dim3 g1(t1, (unsigned)E, chunks), g2(t2, (unsigned)E, chunks * p.slices);
  const bool ua = M % kVec<T> != 0;
  if (four_waves(t1 * touched))
    (ua ? launch_gateup<T, 4, true, NT> : launch_gateup<T, 4, false, NT>)(g1, s, xp, wg, wu, offsets, D, M, ldh, h);
  else
    (ua ? launch_gateup<T, 8, true, NT> : launch_gateup<T, 8, false, NT>)(g1, s, xp, wg, wu, offsets, D, M, ldh, h);
  ABACUS_CHECK_LAUNCH("experts_decode_fwd (gate/up)");
  if (four_waves(t2 * touched))
    hipLaunchKernelGGL((decode_down_kernel<T, 4, NT>), g2, dim3(256), 0, s, (const T*)h, (const T*)wd, offsets, (int)M,
                       (int)D, ldh, R, p.kb_per, p.slices, (T*)y, ws);
  else
    hipLaunchKernelGGL((decode_down_kernel<T, 8, NT>), g2, dim3(512), 0, s, (const T*)h, (const T*)wd, offsets, (int)M,
                       (int)D, ldh, R, p.kb_per, p.slices, (T*)y, ws);
  ABACUS_CHECK_LAUNCH("experts_decode_fwd (down)");
  if (p.slices > 1) {
    const int64_t n = R * D;
    hipLaunchKernelGGL(decode_reduce_kernel<T>, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s, ws, n, p.slices,
                       (T*)y);
    ABACUS_CHECK_LAUNCH("experts_decode_fwd (reduce)");
  }
  return 0;
}

// Shapes taken: up to 16 rows per expert on average in bf16 (E 64 D 2048 M 1408:
// 12 rows 225 -> 186 us, 24 rows 222 either way, 48 rows 239 -> 387, where most
// experts stream their weights twice), 64 in fp32 (E 16 D 1024 M 2816: 64 rows 499 -> 358), tiles no
// wider than the matrices, grid dimensions in range.
bool takes(int64_t R, int64_t D, int64_t M, int64_t E, int dtype) {
  if (dtype != kBF16 && dtype != kF32) return false;
  const int vec = dtype == kBF16 ? 8 : 4, cols = 16 * vec;
  return R >= 1 && E >= 1 && E <= 1024 && D % vec == 0 && D >= cols && M >= cols && D < (1 << 24) && M < (1 << 24) &&
         R <= (dtype == kBF16 ? 16 : 64) * E;
}

// Weights that reach well past what the 256 MB last-level cache can hold from
// one call to the next are read nontemporal.
template <typename T>
int launch_for(const void* xp, const void* wg, const void* wu, const void* wd, const int32_t* offsets, int64_t R,
               int64_t D, int64_t M, int64_t E, int64_t ldh, void* h, void* y, float* ws, hipStream_t s) {
  const int64_t bytes = 3 * std::min(E, R) * D * M * (int64_t)sizeof(T);
  return bytes >= (128ll << 20) ? launch<T, true>(xp, wg, wu, wd, offsets, R, D, M, E, ldh, h, y, ws, s)
                                : launch<T, false>(xp, wg, wu, wd, offsets, R, D, M, E, ldh, h, y, ws, s);
}

}  // namespace
}  // namespace abacus

using namespace abacus;

extern "C" int64_t abacus_experts_decode_ws_bytes(int64_t R, int64_t D, int64_t M, int64_t E, int dtype) {
  if (!takes(R, D, M, E, dtype)) return -1;
  const DownPlan p = plan_down(R, D, M, E, dtype == kBF16 ? kCols<uint16_t> : kCols<float>);
  return p.slices > 1 ? p.slices * R * D * 4 : 0;
}

extern "C" int abacus_experts_decode_fwd(const void* x_perm_RD, const void* w_gate_EDM, const void* w_up_EDM,
                                         const void* w_down_EMD, const int32_t* offsets_E1, int64_t R, int64_t D,
                                         int64_t M, int64_t E, int dtype, int64_t ld_h, void* h, void* y_RD, void* ws,
                                         int64_t ws_bytes, void* stream) {
  const int64_t need = abacus_experts_decode_ws_bytes(R, D, M, E, dtype);
  ABACUS_CHECK_ARG(need >= 0, "experts_decode_fwd: R %lld, D %lld, M %lld, E %lld, dtype %d not taken", (long long)R,
                   (long long)D, (long long)M, (long long)E, dtype);
  const int vec = dtype == kBF16 ? 8 : 4;
  ABACUS_CHECK_ARG(ld_h >= M && ld_h < M + vec && ld_h % vec == 0,
                   "experts_decode_fwd: ld_h %lld must be hidden_dim %lld rounded up to %d", (long long)ld_h,
                   (long long)M, vec);
  ABACUS_CHECK_ARG(x_perm_RD && w_gate_EDM && w_up_EDM && w_down_EMD && offsets_E1 && h && y_RD,
                   "experts_decode_fwd: null pointer");
  ABACUS_CHECK_ARG(ws_bytes >= need && (need == 0 || ws != nullptr), "experts_decode_fwd: workspace of %lld bytes, need %lld",
                   (long long)ws_bytes, (long long)need);
  if (dtype == kBF16)
    return launch_for<uint16_t>(x_perm_RD, w_gate_EDM, w_up_EDM, w_down_EMD, offsets_E1, R, D, M, E, ld_h, h, y_RD,
                            (float*)ws, (hipStream_t)stream);
  return launch_for<float>(x_perm_RD, w_gate_EDM, w_up_EDM, w_down_EMD, offsets_E1, R, D, M, E, ld_h, h, y_RD, (float*)ws,
                       (hipStream_t)stream);
}
