// Expert products of a small forward batch (decode steps, short prompts): few
// routed rows per expert, so the whole cost is streaming the touched experts'
// weights once.
//
// Reference: abacus/moe/moe.py:78-80 (x w_gate, x w_up, (silu(gate) up) w_down
// per expert), as the grouped GEMMs of grouped_gemm.hip; rows are the same
// expert-contiguous rows.
#include <algorithm>
#include <type_traits>

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
// a scalar base plus one of two lane offsets.  HOLD: for a caller without a loop
// around it.
template <typename T, bool UNALIGNED, bool NT, bool HOLD>
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
    const T* wp[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      wp[i] = wb + i * ldw + woff;
      s.w[i] = load_weights<T, UNALIGNED, NT>(wp[i]);
    }
#pragma unroll
    for (int r = 0; r < RG; ++r)
      if ((HOLD && r == 0) || r * kGroup < n_rows) {
#pragma unroll
        for (int v = 0; v < S::XV; ++v) s.x[r][v] = ld16(xb + v * kVec<T> + xoff[r]);
      }
    // The addresses outlive their loads: else the compiler forms them in the loads' own destinations,
    // which waits for the loads still in flight there (E 64 D 2048 M 1408, 64 tokens: 205 -> 231 us).
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if constexpr (HOLD) asm volatile("" : : "v"(wp[i]));
  };
  auto use = [&](const S& s) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < RG; ++r)
      if ((HOLD && r == 0) || r * kGroup < n_rows) step_mfma(acc[r], s.w, s.x[r]);
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

// Tiles numbered over the rows that exist: (expert, columns, rows), ROWS rows each and
// the rows fastest, an expert's first SKIP row tiles not counted.  Block b takes
// its tile from an equal contiguous share for each XCD (it runs on XCD b % 8), so
// that the blocks that read the same weights run beside each other on one L2.
// Every wave finds the tile by itself; false: this block has none.
struct RowTile {
  int e, row0, row1, col;  // row1: the expert's end or row0 + ROWS
};
template <int ROWS, int SKIP>
__device__ __forceinline__ bool row_tile(const int32_t* __restrict__ offsets, int E, int cols, int b, int lane,
                                         RowTile& t) {
  auto chunks = [&](int e) { return e < E ? max(0, (offsets[e + 1] - offsets[e] + ROWS - 1) / ROWS - SKIP) : 0; };
  int total = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    int c = chunks(e0 + lane);
#pragma unroll
    for (int o = 32; o; o >>= 1) c += __shfl_xor(c, o, 64);
    total += __builtin_amdgcn_readfirstlane(c);
  }
  const int per = (total * cols + 7) / 8;
  const int L = (b & 7) * per + (b >> 3);
  if ((b >> 3) >= per || L >= total * cols) return false;
  int before = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int c = chunks(e0 + lane);
    int end = c;  // inclusive scan over the lanes
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(end, o, 64);
      if (lane >= o) end += u;
    }
    const uint64_t past = __ballot((before + end) * cols > L);
    if (past) {
      const int l = __builtin_ctzll(past);
      const int n = __builtin_amdgcn_readlane(c, l);
      const int at = L - (before + __builtin_amdgcn_readlane(end, l) - n) * cols;
      t.e = e0 + l;
      t.col = at / n;
      t.row0 = offsets[t.e] + (at % n + SKIP) * ROWS;
      t.row1 = min(t.row0 + ROWS, offsets[t.e + 1]);
      return true;
    }
    before += __builtin_amdgcn_readlane(end, 63);
  }
  return false;
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

// This block's tile of up to kRows rows.  First a block for each (expert, columns), which
// takes the expert's first kRows rows: all there is where routing is even.  After
// them (`more`) come the numbered tiles of the rows past those, as many blocks as
// R / kRows row tiles need, wherever the rows are: one expert may hold all of them.
// MANY (more than 8 rows per expert on average): those blocks read the weights, which
// the blocks beside them read too, through the caches.  It costs the others 3-4%, as two
// streams share the registers, so a smaller batch reads all of them in the one way.
// us with at most four passes of an expert side by side -> here, every token on the same
// experts, beside the 256-row tiles: bf16 E 128 D 1024 M 2816, 2048 tokens top-1 1077 ->
// 160 (149), E 64 D 2048 M 1408, 170 tokens top-6 191 -> 108 (112), 64 tokens 113 -> 117 (87); fp32
// E 64 D 1024 M 1408, 4096 tokens top-1 2816 -> 424 (537).  The second and the last of them
// with even routing 221 -> 231 (259), 660 -> 588 (705), Zipf-skewed 260 -> 246 (239), 1363 -> 484 (696).
__device__ __forceinline__ bool block_tile(const int32_t* __restrict__ offsets, int E, int cols, int lane, RowTile& t,
                                           bool& more) {
  more = (int)blockIdx.y >= E;
  if (more) return row_tile<kRows, 1>(offsets, E, cols, ((int)blockIdx.y - E) * cols + (int)blockIdx.x, lane, t);
  t.e = blockIdx.y;
  t.col = blockIdx.x;
  t.row0 = offsets[t.e];
  t.row1 = min(t.row0 + kRows, offsets[t.e + 1]);
  return t.row0 < t.row1;
}
// Its grid: (columns, experts, then whole turns of the 8 XCDs for R / kRows row tiles).
int64_t grid_rows(int64_t R, int64_t E, int64_t cols) { return E + (R > kRows ? R / kRows + (7 + cols - 1) / cols : 0); }

// H = silu(x w_gate) (x w_up) for one expert's rows and kCols columns per
// block.  The first half of the W waves share w_gate's k-blocks, the second
// half w_up's; the partial products meet in LDS and are added in wave order.
template <typename T, int W, bool UNALIGNED, bool NT, bool MANY>
__global__ __launch_bounds__(W * 64, 2) void decode_gateup_kernel(const T* __restrict__ xp,
                                                                    const T* __restrict__ w_gate,
                                                                    const T* __restrict__ w_up,
                                                                    const int32_t* __restrict__ offsets, int E, int D,
                                                                    int M, int64_t ldh, T* __restrict__ h) {
  constexpr int HW = W / 2;  // waves per matrix
  constexpr int NC = kCols<T>, PART = kGroup * NC;
  __shared__ __attribute__((aligned(16))) float part[W * PART];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave / HW;
  const int cols = (M + NC - 1) / NC;
  RowTile tile;
  bool more;
  if (!block_tile(offsets, E, cols, lane, tile, more)) return;
  const int row1 = tile.row1;
  const int n0 = min(tile.col * NC, M - NC);  // the last tile overlaps its neighbour: the same sums, written twice
  const T* w = (half ? w_up : w_gate) + (int64_t)tile.e * D * M + n0;
  auto pass = [&](int r0) __attribute__((always_inline)) {
    dec_f32x4 acc[RG][kVec<T>] = {};
    auto stream = [&](auto nt) __attribute__((always_inline)) {
      stream_rows<T, UNALIGNED, decltype(nt)::value, MANY>(w, M, xp + (int64_t)r0 * D, D, row1 - r0, D, wave % HW,
                                                     (D + kKB - 1) / kKB, HW, lane, acc);
    };
    if (!(MANY && NT && more)) stream(std::bool_constant<NT>{});
    else if constexpr (MANY && NT) stream(std::false_type{});
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
      if (tile.col == cols - 1 && tid < kGroup && rg0 + tid < row1)  // H's pad columns
        for (int64_t c = M; c < ldh; ++c) h[(int64_t)(rg0 + tid) * ldh + c] = (T)0;
    }
  };
  if constexpr (MANY) {
    pass(tile.row0);
  } else {
    int step = kRows;  // one pass, in a loop as far as the compiler knows: it then keeps the addresses apart
    asm("" : "+s"(step));
    for (int r0 = tile.row0; r0 < row1; r0 += step) pass(r0);
  }
}

// Y = H w_down for one expert's rows, kCols columns and one slice of the
// k-blocks per block, shared by its W waves.  One slice: Y itself; more: fp32
// partials [slice][R][D] for decode_reduce_kernel.
template <typename T, int W, bool NT, bool MANY>
__global__ __launch_bounds__(W * 64, 2) void decode_down_kernel(const T* __restrict__ h, const T* __restrict__ w_down,
                                                                  const int32_t* __restrict__ offsets, int E, int M,
                                                                  int D, int64_t ldh, int64_t R, int kb_per, int slices,
                                                                  T* __restrict__ y, float* __restrict__ ws) {
  constexpr int NC = kCols<T>, PART = kGroup * NC;
  __shared__ __attribute__((aligned(16))) float part[W * PART];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  RowTile tile;
  bool more;
  if (!block_tile(offsets, E, (D + NC - 1) / NC, lane, tile, more)) return;
  const int row1 = tile.row1;
  const int n0 = min(tile.col * NC, D - NC);
  const int nkb = (M + kKB - 1) / kKB, slice = (int)blockIdx.z, kb0 = slice * kb_per, kb1 = min(kb0 + kb_per, nkb);
  const T* w = w_down + (int64_t)tile.e * M * D + n0;
  auto pass = [&](int r0) __attribute__((always_inline)) {
    dec_f32x4 acc[RG][kVec<T>] = {};
    auto stream = [&](auto nt) __attribute__((always_inline)) {
      stream_rows<T, false, decltype(nt)::value, MANY>(w, D, h + (int64_t)r0 * ldh, ldh, row1 - r0, M, kb0 + wave, kb1, W,
                                                 lane, acc);
    };
    if (!(MANY && NT && more)) stream(std::bool_constant<NT>{});
    else if constexpr (MANY && NT) stream(std::false_type{});
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
  };
  if constexpr (MANY) {
    pass(tile.row0);
  } else {
    int step = kRows;
    asm("" : "+s"(step));
    for (int r0 = tile.row0; r0 < row1; r0 += step) pass(r0);
  }
}

// More rows per expert (bf16): blocks of up to 64 rows of one expert, so that
// most experts' weights still stream once, numbered as row_tile does (weights that
// are read nontemporal miss the L2 there: E 64 D 2048 M 1408, 682 tokens 346 -> 410 us).
// What bounds them is the weight stream as long as an expert's rows are one block's.
// 64 rows: more would not fit the registers (128 of 256 hold the sums), fewer stream
// the weights more often.
constexpr int kMidRows = 64;

// acc[r][j] += step_mfma's product for G groups of 16 rows, each column transposed once.
template <int G>
__device__ inline void step_groups(dec_f32x4 (&acc)[G][8], const Vec16 (&w)[8], const Vec16 (&x)[G]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    Vec16 b;
#pragma unroll
    for (int p = 0; p < 4; ++p)
      b.w[p] = __builtin_amdgcn_perm(w[2 * p + 1].w[j >> 1], w[2 * p].w[j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
#pragma unroll
    for (int r = 0; r < G; ++r)
      acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dec_bf16x8, x[r]),
                                                          __builtin_bit_cast(dec_bf16x8, b), acc[r][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);  // one column's transpose live at a time
  }
}

// A wave-uniform pointer kept in scalar registers, for loops whose accumulators
// leave no room: else the compiler steps one 64-bit vector address per load
// through the loop, some 50 registers (64 rows a pass then spill in it).
typedef const __attribute__((address_space(1))) char* global_bytes;
__device__ inline global_bytes scalar_base(const void* p) {
  uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uint64_t)p);
  uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)p >> 32));
  asm("" : "+s"(lo), "+s"(hi));
  return (global_bytes)(((uint64_t)hi << 32) | lo);
}
// The 16 bytes at base + off, aligned or at any element.
template <bool UNALIGNED>
__device__ inline Vec16 load_at(global_bytes base, uint32_t off) {
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  typedef uint32_t u32x4_ua __attribute__((ext_vector_type(4), aligned(2)));
  typedef const __attribute__((address_space(1))) u32x4_t* whole_ptr;
  typedef const __attribute__((address_space(1))) u32x4_ua* any_ptr;
  u32x4_t v;
  if constexpr (UNALIGNED) {
    v = *(any_ptr)(base + off);
  } else {
    v = *(whole_ptr)(base + off);
  }
  Vec16 r;
  r.w[0] = v.x; r.w[1] = v.y; r.w[2] = v.z; r.w[3] = v.w;
  return r;
}

// acc += x[rows] * w over the k-blocks kb0, kb0 + kstride, ... < kb1, as
// stream_rows, for G groups of rows that are all computed (no branches between
// the loads and products), the weights at any element.
template <bool UNALIGNED, int G>
__device__ __forceinline__ void stream_groups(const uint16_t* __restrict__ w, int64_t ldw, const uint16_t* __restrict__ x,
                                              int64_t pitch, int n_rows, int K, int kb0, int kb1, int kstride, int lane,
                                              dec_f32x4 (&acc)[G][8]) {
  struct Operands {
    Vec16 w[8], x[G];
  };
  const int kl = 8 * (lane >> 4);
  const uint32_t woff = 2 * ((uint32_t)kl * (uint32_t)ldw + 8 * (lane & 15));  // bytes
  uint32_t xoff[G];
#pragma unroll
  for (int r = 0; r < G; ++r) xoff[r] = 2 * ((uint32_t)min(r * kGroup + (lane & 15), n_rows - 1) * (uint32_t)pitch + kl);
  auto load = [&](Operands& s, int kb) __attribute__((always_inline)) {
    const uint16_t* wb = w + (int64_t)kb * kKB * ldw;
#pragma unroll
    for (int i = 0; i < 8; ++i) s.w[i] = load_at<UNALIGNED>(scalar_base(wb + i * ldw), woff);
    const global_bytes xb = scalar_base(x + (int64_t)kb * kKB);
#pragma unroll
    for (int r = 0; r < G; ++r) s.x[r] = load_at<false>(xb, xoff[r]);
  };
  const int whole = min(kb1, K / kKB);  // k-blocks without a tail
  Operands a, b;
  int kb = kb0;
  if (kb < whole) load(a, kb);
  while (kb < whole) {  // the next block's loads go out before this one's products
    if (kb + kstride < whole) load(b, kb + kstride);
    step_groups<G>(acc, a.w, a.x);
    kb += kstride;
    if (kb >= whole) break;
    if (kb + kstride < whole) load(a, kb + kstride);
    step_groups<G>(acc, b.w, b.x);
    kb += kstride;
  }
  if (kb < kb1) {  // the tail block: rows from K on read row K - 1 and count as zero
    const int k = kb * kKB + kl;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      a.w[i] = load_weights<uint16_t, UNALIGNED, false>(w + (int64_t)min(k + i, K - 1) * ldw + 8 * (lane & 15));
      if (k + i >= K) a.w[i] = zero16();
    }
#pragma unroll
    for (int r = 0; r < G; ++r) a.x[r] = k < K ? ld16(x + (int64_t)kb * kKB + xoff[r] / 2) : zero16();
    step_groups<G>(acc, a.w, a.x);
  }
}

// H = silu(x w_gate) (x w_up) for rows r0 .. min(r0 + 16 G, row1) - 1 of one
// expert and the kCols columns from n0.  The first half of the block's W waves
// share w_gate's k-blocks, the second half w_up's (w: this wave's matrix at n0);
// the partial products meet in LDS and are added in wave order.  pads: this
// block also writes H's pad columns.
template <int W, int G>
__device__ __forceinline__ void mid_gateup_pass(float* part, const uint16_t* __restrict__ w, const uint16_t* __restrict__ xp, int r0, int row1, int n0,
                                   bool pads, int D, int M, int64_t ldh, uint16_t* __restrict__ h, int tid) {
  constexpr int HW = W / 2;  // waves per matrix
  constexpr int NC = kCols<uint16_t>, PART = kGroup * NC;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  dec_f32x4 acc[G][8] = {};
  stream_groups<true, G>(w, M, xp + (int64_t)r0 * D, D, row1 - r0, D, wave % HW, (D + kKB - 1) / kKB, HW, lane, acc);
#pragma unroll
  for (int r = 0; r < G; ++r) {
    const int rg0 = r0 + r * kGroup;
    if (rg0 >= row1) break;
    __syncthreads();  // the previous group's sums are read
    store_partial<uint16_t>(part + wave * PART, acc[r], lane);
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
        const float g = round_to<uint16_t>(s[0][i]), u = round_to<uint16_t>(s[1][i]);
        o[i] = round_to<uint16_t>(silu_f32(g)) * u;
      }
      store4<uint16_t>(h + (int64_t)row * ldh + n0 + c, o[0], o[1], o[2], o[3]);
    }
    if (pads && tid < kGroup && rg0 + tid < row1)
      for (int64_t c = M; c < ldh; ++c) h[(int64_t)(rg0 + tid) * ldh + c] = 0;
  }
}

// Y = H w_down for rows r0 .. min(r0 + 16 G, row1) - 1 of one expert, the
// kCols columns from n0 and the k-blocks kb0 .. kb1 - 1, shared by the block's W
// waves.  One slice: Y itself; more: fp32 partials [slice][R][D] for
// decode_reduce_kernel.
template <int W, int G>
__device__ __forceinline__ void mid_down_pass(float* part, const uint16_t* __restrict__ w, const uint16_t* __restrict__ h, int r0, int row1, int n0,
                                 int M, int D, int64_t ldh, int64_t R, int kb0, int kb1, int slice, int slices,
                                 uint16_t* __restrict__ y, float* __restrict__ ws, int tid) {
  constexpr int NC = kCols<uint16_t>, PART = kGroup * NC;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  dec_f32x4 acc[G][8] = {};
  stream_groups<false, G>(w, D, h + (int64_t)r0 * ldh, ldh, row1 - r0, M, kb0 + wave, kb1, W, lane, acc);
#pragma unroll
  for (int r = 0; r < G; ++r) {
    const int rg0 = r0 + r * kGroup;
    if (rg0 >= row1) break;
    __syncthreads();
    store_partial<uint16_t>(part + wave * PART, acc[r], lane);
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
      if (slices == 1) store4<uint16_t>(y + (int64_t)row * D + n0 + c, t.x, t.y, t.z, t.w);
      else *reinterpret_cast<float4*>(ws + ((int64_t)slice * R + row) * D + n0 + c) = t;
    }
  }
}

__global__ __launch_bounds__(256, 2) void mid_gateup_kernel(const uint16_t* __restrict__ xp,
                                                            const uint16_t* __restrict__ w_gate,
                                                            const uint16_t* __restrict__ w_up,
                                                            const int32_t* __restrict__ offsets, int E, int D, int M,
                                                            int64_t ldh, uint16_t* __restrict__ h) {
  constexpr int NC = kCols<uint16_t>;
  __shared__ __attribute__((aligned(16))) float part[4 * kGroup * NC];
  const int tid = threadIdx.x, cols = (M + NC - 1) / NC;
  RowTile t;
  if (!row_tile<kMidRows, 0>(offsets, E, cols, (int)blockIdx.x, tid & 63, t)) return;
  const int half = __builtin_amdgcn_readfirstlane(tid >> 7), n0 = min(t.col * NC, M - NC);
  const uint16_t* w = (half ? w_up : w_gate) + (int64_t)t.e * D * M + n0;
  const bool pads = t.col == cols - 1;
  if (t.row1 - t.row0 > kRows)
    mid_gateup_pass<4, kMidRows / kGroup>(part, w, xp, t.row0, t.row1, n0, pads, D, M, ldh, h, tid);
  else
    mid_gateup_pass<4, RG>(part, w, xp, t.row0, t.row1, n0, pads, D, M, ldh, h, tid);
}

__global__ __launch_bounds__(256, 2) void mid_down_kernel(const uint16_t* __restrict__ h,
                                                          const uint16_t* __restrict__ w_down,
                                                          const int32_t* __restrict__ offsets, int E, int M, int D,
                                                          int64_t ldh, int64_t R, int kb_per, uint16_t* __restrict__ y,
                                                          float* __restrict__ ws) {
  constexpr int NC = kCols<uint16_t>;
  __shared__ __attribute__((aligned(16))) float part[4 * kGroup * NC];
  const int tid = threadIdx.x, slice = (int)blockIdx.y, slices = (int)gridDim.y;
  RowTile t;
  if (!row_tile<kMidRows, 0>(offsets, E, (D + NC - 1) / NC, (int)blockIdx.x, tid & 63, t)) return;
  const int n0 = min(t.col * NC, D - NC);
  const int kb0 = slice * kb_per, kb1 = min(kb0 + kb_per, (M + kKB - 1) / kKB);
  const uint16_t* w = w_down + (int64_t)t.e * M * D + n0;
  if (t.row1 - t.row0 > kRows)
    mid_down_pass<4, kMidRows / kGroup>(part, w, h, t.row0, t.row1, n0, M, D, ldh, R, kb0, kb1, slice, slices,
                                                  y, ws, tid);
  else
    mid_down_pass<4, RG>(part, w, h, t.row0, t.row1, n0, M, D, ldh, R, kb0, kb1, slice, slices, y, ws, tid);
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

template <typename T, int W, bool UNALIGNED, bool NT, bool MANY>
void launch_gateup(dim3 grid, hipStream_t s, const void* xp, const void* wg, const void* wu, const int32_t* offsets,
                   int64_t E, int64_t D, int64_t M, int64_t ldh, void* h) {
  hipLaunchKernelGGL((decode_gateup_kernel<T, W, UNALIGNED, NT, MANY>), grid, dim3(W * 64), 0, s, (const T*)xp,
                     (const T*)wg, (const T*)wu, offsets, (int)E, (int)D, (int)M, ldh, (T*)h);
}

template <typename T>
int launch_reduce(const float* ws, int64_t n, int slices, void* y, hipStream_t s) {
  if (slices <= 1) return 0;
  hipLaunchKernelGGL(decode_reduce_kernel<T>, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s, ws, n, slices, (T*)y);
  ABACUS_CHECK_LAUNCH("experts_decode_fwd (reduce)");
  return 0;
}

// Rows per expert from which the blocks of 64 rows run (taken for unaligned
// hidden sizes only).
bool mid_rows(int64_t R, int64_t E, int dtype) { return dtype == kBF16 && R > 16 * E; }

int launch_mid(const void* xp, const void* wg, const void* wu, const void* wd, const int32_t* offsets, int64_t R, int64_t D,
               int64_t M, int64_t E, int64_t ldh, void* h, void* y, float* ws, hipStream_t s) {
  constexpr int NC = kCols<uint16_t>;
  const int64_t tiles = R / kMidRows + std::min(E, R);  // at most, and whole turns of the 8 XCDs
  const int64_t t1 = (tiles * ((M + NC - 1) / NC) + 7) / 8 * 8, t2 = (tiles * ((D + NC - 1) / NC) + 7) / 8 * 8;
  const DownPlan p = plan_down(R, D, M, E, NC);
  hipLaunchKernelGGL(mid_gateup_kernel, dim3((unsigned)t1), dim3(256), 0, s, (const uint16_t*)xp, (const uint16_t*)wg,
                     (const uint16_t*)wu, offsets, (int)E, (int)D, (int)M, ldh, (uint16_t*)h);
  ABACUS_CHECK_LAUNCH("experts_decode_fwd (gate/up)");
  hipLaunchKernelGGL(mid_down_kernel, dim3((unsigned)t2, (unsigned)p.slices), dim3(256), 0, s, (const uint16_t*)h,
                     (const uint16_t*)wd, offsets, (int)E, (int)M, (int)D, ldh, R, p.kb_per, (uint16_t*)y, ws);
  ABACUS_CHECK_LAUNCH("experts_decode_fwd (down)");
  return launch_reduce<uint16_t>(ws, R * D, p.slices, y, s);
}

template <typename T, bool NT, bool MANY>
int launch(const void* xp, const void* wg, const void* wu, const void* wd, const int32_t* offsets, int64_t R, int64_t D,
           int64_t M, int64_t E, int64_t ldh, void* h, void* y, float* ws, hipStream_t s) {
  constexpr int NC = kCols<T>;
  const int64_t t1 = (M + NC - 1) / NC, t2 = (D + NC - 1) / NC, touched = std::min(E, R);
  const DownPlan p = plan_down(R, D, M, E, NC);
  const dim3 g1((unsigned)t1, (unsigned)grid_rows(R, E, t1));
  const dim3 g2((unsigned)t2, (unsigned)grid_rows(R, E, t2), (unsigned)p.slices);
  const bool ua = M % kVec<T> != 0;
  if (four_waves(t1 * touched))
    (ua ? launch_gateup<T, 4, true, NT, MANY> : launch_gateup<T, 4, false, NT, MANY>)(g1, s, xp, wg, wu, offsets, E, D, M, ldh, h);
  else
    (ua ? launch_gateup<T, 8, true, NT, MANY> : launch_gateup<T, 8, false, NT, MANY>)(g1, s, xp, wg, wu, offsets, E, D, M, ldh, h);
  ABACUS_CHECK_LAUNCH("experts_decode_fwd (gate/up)");
  if (four_waves(t2 * touched))
    hipLaunchKernelGGL((decode_down_kernel<T, 4, NT, MANY>), g2, dim3(256), 0, s, (const T*)h, (const T*)wd, offsets,
                       (int)E, (int)M, (int)D, ldh, R, p.kb_per, p.slices, (T*)y, ws);
  else
    hipLaunchKernelGGL((decode_down_kernel<T, 8, NT, MANY>), g2, dim3(512), 0, s, (const T*)h, (const T*)wd, offsets,
                       (int)E, (int)M, (int)D, ldh, R, p.kb_per, p.slices, (T*)y, ws);
  ABACUS_CHECK_LAUNCH("experts_decode_fwd (down)");
  return launch_reduce<T>(ws, R * D, p.slices, y, s);
}

// bf16 hidden sizes that are not whole vectors: the tiles of grouped_gemm.hip
// need every weight copied to an aligned pitch first, so the weights are streamed as
// they are up to 128 rows per expert on average.  Eval layer, copies + tiles against
// this (us): E 64 D 2048 M 1406 top-6, 513 tokens 549 -> 310 (skewed routing 554 -> 332), 1366
// tokens 617 -> 500; E 8 D 4096 M 14330, 68 tokens 1180 -> 548, 512 tokens 1270 -> 1118, 768 tokens
// (192 rows per expert) 1359 -> 1392; E 16 D 1024 M 2730, 136 tokens 156 -> 82, 1024 tokens 195 ->
// 164.  Whole vectors stay with the tiles: E 64 D 2048 M 1408, 512 tokens 276 against 299 here.
constexpr int kMidMax = 128;

// Shapes taken: up to 16 rows per expert on average in bf16 (E 64 D 2048 M 1408:
// 12 rows 225 -> 186 us, 24 rows 222 either way, 48 rows 239 -> 387, where most
// experts stream their weights twice), 64 in fp32 (E 16 D 1024 M 2816: 64 rows 499 -> 358), tiles no
// wider than the matrices, grid dimensions in range.
bool takes(int64_t R, int64_t D, int64_t M, int64_t E, int dtype) {
  if (dtype != kBF16 && dtype != kF32) return false;
  const int vec = dtype == kBF16 ? 8 : 4, cols = 16 * vec;
  return R >= 1 && E >= 1 && E <= 1024 && D % vec == 0 && D >= cols && M >= cols && D < (1 << 24) && M < (1 << 24) &&
         R <= (dtype == kF32 ? 64 : M % vec == 0 ? 16 : kMidMax) * E;
}

// Weights that reach well past what the 256 MB last-level cache can hold from
// one call to the next are read nontemporal.
template <typename T>
int launch_for(const void* xp, const void* wg, const void* wu, const void* wd, const int32_t* offsets, int64_t R,
               int64_t D, int64_t M, int64_t E, int64_t ldh, void* h, void* y, float* ws, hipStream_t s) {
  if (mid_rows(R, E, sizeof(T) == 2 ? kBF16 : kF32)) return launch_mid(xp, wg, wu, wd, offsets, R, D, M, E, ldh, h, y, ws, s);
  const int64_t bytes = 3 * std::min(E, R) * D * M * (int64_t)sizeof(T);
  const bool nt = bytes >= (128ll << 20), many = R > 8 * E;  // (see block_tile)
  const auto run = nt ? (many ? launch<T, true, true> : launch<T, true, false>)
                      : (many ? launch<T, false, true> : launch<T, false, false>);
  return run(xp, wg, wu, wd, offsets, R, D, M, E, ldh, h, y, ws, s);
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
