// Token logprobs straight from hidden states and the output (LM-head) weight:
// the logits tile H[rows] . W[cols]^T is formed on the MFMA units and reduced
// in the same kernel, so the [T, V] logits are never written.
//
// Semantics follow nemo_rl/distributed/model_utils.py:2541-2745
// (from_parallel_hidden_states_to_logprobs, ChunkedDistributedHiddenStatesToLogprobs)
// with a vocab group of size 1:
//   logits    = bf16(H . W^T)                (the reference's bf16 matmul output)
//   logprob_t = (x_t - m) - log(sum_v exp(x_v - m)),  0 for targets outside [vs, ve)
//   backward  G = (onehot(t) - softmax(x)) * g,  dH = G . W,  dW = G^T . H
// The forward kernel writes, per row and per 256-column tile, the tile's
// (max, sum exp(x - max)) and the target logit; a merge kernel combines the
// tiles of a row.  The gradient kernel recomputes a logits tile and writes the
// bf16 G tile and its transpose; the two products that consume G run on the
// same tile loop as a plain GEMM.  Row counts may live on the device (the
// backward's active rows): the kernels read them and skip what lies past them,
// so the host never waits for them.
//
// Tile: 256 rows x 256 columns per 256-thread workgroup.  Each wave owns a
// 128 x 128 quarter as 8 x 8 v_mfma_f32_16x16x32 tiles (256 fp32 accumulators
// per lane).  The hidden dimension streams through two LDS stages
// of 64 elements (64 KB each: 256 rows of H and 256 rows of W, 128 B per row),
// filled by direct global->LDS loads (buffer_load_dwordx4 ... lds) one stage
// ahead of the MFMAs: no staging registers and no LDS store instructions sit
// between the loads and the MFMAs, and the only waits are one vmcnt + barrier
// per stage.  Each row of a stage is one 128-byte line of H or W.  A row's
// eight 16-byte chunks are XOR-swizzled by (row / 2) % 8 (see lds_off), so the
// 16 rows read by one pass of an MFMA operand load fall in distinct banks.
//
// The MFMA lane layouts (checked on gfx950) stand at Mma<E>.

#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.h"

#pragma clang fp contract(off)

namespace mirl {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Operand dtype of the tile loop: its fragment (16 bytes of a row per lane), the
// MFMA tile of kT x kT outputs and its accumulator.  run(w, h, c) forms
// c += W . H^T, W's rows along the accumulator's first index.
//
// 16-bit operands: v_mfma_f32_16x16x32.  Lane l holds elements k = (l / 16) * 8 + 0..7
// of row l % 16 of either operand, and accumulator element v of lane l is
// [W row (l / 16) * 4 + v][H row l % 16]: four consecutive vocabulary columns of one
// logits row.  (v_mfma_f32_32x32x16 does the same work per cycle with half the
// instructions, but the chip runs slower under it: forward of [16384, 4096] x
// [151808, 4096] 15.3 ms against 14.6 with the same epilogue.  Four columns per lane
// make the epilogue's LDS writes 8-byte pieces and its row data one set per eight
// tiles, and the plain GEMM's stores 8- or 16-byte pieces: forward 14.0 ms, 1450
// TFLOP/s; gradient 6.85 -> 6.1 ms of 5888 rows; dW 6.4 -> 5.65; dH 6.1 -> 5.65.)
template <class E>
struct Mma;
template <>
struct Mma<BF16> {
  typedef __bf16 frag __attribute__((ext_vector_type(8)));
  typedef f32x4 acc_t;
  static constexpr int kT = 16;
  __device__ __forceinline__ static f32x4 run(frag w, frag h, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, h, c, 0, 0, 0);
  }
};
template <>
struct Mma<F16> {
  typedef _Float16 frag __attribute__((ext_vector_type(8)));
  typedef f32x4 acc_t;
  static constexpr int kT = 16;
  __device__ __forceinline__ static f32x4 run(frag w, frag h, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(w, h, c, 0, 0, 0);
  }
};
// fp32 operands (plain GEMM only): the planes of a tile go through 32 x 32 outputs
// (see the kernel), and so do the tiles that the planes do not cover: a 16-byte
// fragment holds four hidden elements of a row, k = (l / 32) * 4 + 0..3, and feeds
// four v_mfma_f32_32x32x2_f32, element e of both fragments to the e-th one.  That
// instruction takes A[l % 32][l / 32] and B[l / 32][l % 32] from lane l, so the
// four together sum the products over the fragment's eight hidden elements
// (element e of the lanes below 32 is k = e, of the others k = 4 + e).
// Accumulator element v of lane l is
// [W row (v / 4) * 8 + (l / 32) * 4 + v % 4][H row l % 32].
template <>
struct Mma<F32> {
  typedef float frag __attribute__((ext_vector_type(4)));
  typedef f32x16 acc_t;
  static constexpr int kT = 32;
  __device__ __forceinline__ static f32x16 run(frag w, frag h, f32x16 c) {
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(w[0], h[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(w[1], h[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(w[2], h[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(w[3], h[3], c, 0, 0, 0);
    return c;
  }
};

// 16-bit element bits <-> fp32 for a dtype E (round to nearest even).
template <class E>
__device__ __forceinline__ uint16_t bits_of(float f) {
  return __builtin_bit_cast(uint16_t, E::from_float(f));
}
template <class E>
__device__ __forceinline__ float value_of(uint16_t b) {
  return E::load_raw(__builtin_bit_cast(typename E::raw, b));
}
// Four fp32 values rounded to E, packed.
template <class E>
__device__ __forceinline__ uint2 pack4(f32x4 o) {
  if constexpr (std::is_same<E, BF16>::value)
    return uint2{BF16::pack2(o[0], o[1]), BF16::pack2(o[2], o[3])};
  else
    return uint2{(uint32_t)bits_of<E>(o[0]) | ((uint32_t)bits_of<E>(o[1]) << 16),
                 (uint32_t)bits_of<E>(o[2]) | ((uint32_t)bits_of<E>(o[3]) << 16)};
}
typedef __attribute__((address_space(3))) void* lds_ptr_t;

constexpr int kBM = 256;                 // rows per tile
constexpr int kBN = 256;                 // vocabulary columns per tile
constexpr int kSK = 64;                  // 16-bit hidden elements per LDS stage (128 bytes)
constexpr int kStages = 2;
constexpr int kThreads = 256;            // 4 waves in a 2 x 2 arrangement
constexpr int kWaves = kThreads / kWave;
constexpr int kWM = 128, kWN = 128;      // per-wave quarter
constexpr int kRowBytes = kSK * 2;       // 128 B: one tile row of a stage
constexpr int kHalfBytes = kBM * kRowBytes;    // 32 KB: the H (or W) rows of a stage
constexpr int kStageBytes = 2 * kHalfBytes;    // 64 KB
constexpr int kDmaBytes = kWave * 16;          // one direct load: 64 lanes x 16 B = 8 rows
constexpr int kDmaRows = kDmaBytes / kRowBytes;
constexpr int kDmaPerWave = kHalfBytes / kDmaBytes / kWaves;  // loads of H (and of W) per wave and stage
constexpr int kEpiRows = kStageBytes / (kBN * 2);  // epilogue tile rows held by one stage array
constexpr int kGroupM = 8;               // row tiles sharing a sweep over the vocabulary
constexpr int kXcds = 8;                 // accelerator dies, each with its own L2
static_assert(kBM == kBN, "H and W halves of a stage have the same size");
static_assert(kEpiRows * kStages == kBM, "the epilogue tile fills the stage arrays");
static_assert(kEpiRows == kWM, "a wave's epilogue rows live in one stage array");

// LDS byte offset (within a stage half) of 16-byte chunk `chunk` of tile row
// `row`.  A ds_read_b128 serves 16 lanes per pass (16 x 16 B = the 64
// four-byte banks); an MFMA operand read has those lanes on 16 consecutive rows
// at one chunk.  Two 128-byte rows span the 64 banks, so the chunk is XOR-ed
// with (row / 2) % 8: the 8 even and the 8 odd rows then each hit 8 distinct
// chunks, i.e. 16 distinct bank groups.
__device__ __forceinline__ int lds_off(int row, int chunk) {
  return row * kRowBytes + ((chunk ^ ((row >> 1) & 7)) << 4);
}

// Epilogue layout of the [256][256] bf16 tile: row r lives in stage array
// r / 128 at local row r % 128, row-major, 16-byte chunks XOR-swizzled by xs_swizzle(r)
// (element index within the array).  16 consecutive rows at one chunk (the
// accumulators' writes, the forward's row walk) and 8 rows 8 apart at two chunks (the
// transposed read) each fall in distinct banks.
__device__ __forceinline__ int xs_swizzle(int row) { return (row ^ (row >> 3)) & 31; }
__device__ __forceinline__ int xs_index(int row, int col) {
  return (row & (kEpiRows - 1)) * kBN + ((((col >> 3) ^ xs_swizzle(row)) << 3) | (col & 7));
}

// s_waitcnt vmcnt(N) lgkmcnt(0), then s_barrier.  The memory clobber keeps the
// compiler from moving LDS accesses across the barrier.
template <int N>
__device__ __forceinline__ void wait_vm_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// The low bf16 of a pair, widened.  By a byte permute: for a shift, the compiler would
// form the low half once more with a conversion of its own.
__device__ __forceinline__ float low_bf16(uint32_t w) {
  return __uint_as_float(__builtin_amdgcn_perm(0u, w, 0x01000c0cu));
}

// w | the bits of a and b.  In asm: the compiler would gather the values to join first,
// on the stack.
__device__ __forceinline__ uint32_t or3(uint32_t w, float a, float b) {
  asm("v_or3_b32 %0, %0, %1, %2" : "+v"(w) : "v"(a), "v"(b));
  return w;
}

// A value that every lane of the wave holds, in scalar registers.
__device__ __forceinline__ int64_t uniform(int64_t x) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)x);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)x >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// f(integral_constant<int, 0>) .. f(integral_constant<int, N - 1>): a loop whose index
// the body may use in a constant expression.
template <int... I, class F>
__device__ __forceinline__ void static_for_(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_(std::make_integer_sequence<int, N>{}, f);
}

enum LceMode { kFwd = 0, kGrad = 1, kGemm = 2 };

struct LceParams {
  const void* h;  // [T, Hd] of the kernel's E (bf16, fp16; fp32 for the plain GEMM), row stride ldh
  const void* w;  // [V, Hd] of the same dtype, row stride ldw
  int64_t ldh, ldw;
  int64_t V, Hd;
  int64_t row0, nrows;  // rows handled: [row0, row0 + nrows)
  int64_t bsz;          // row r is (s, b) = (r / bsz, r % bsz)
  const int64_t* target;
  int64_t tsb, tss;
  int64_t vs, ve;
  int64_t n_mt, n_nt;   // row tiles, column tiles
  // forward
  float* part;          // [nrows, n_nt, 2]
  float* xt;            // [nrows]
  // gradient
  const float* stats;   // [T, 2] {max, logsum} by absolute row
  const float* g;
  int64_t gsb, gss;
  uint16_t* G;          // [nrows, V] bf16, row stride ldg
  int64_t ldg;
  uint16_t* Gt;         // or null: G transposed, [V, ldgt] bf16 (column r - row0 of row v)
  int64_t ldgt;
  // plain GEMM (kGemm): C = A . B^T with A = h [nrows, Hd], B = w [V, Hd]; the
  // hidden dimension is split into n_ks ranges of kb_len (C holds n_ks
  // partial products [n_ks][nrows][ldc]), or Cb receives bf16(C) (n_ks = 1)
  int64_t n_ks, kb_len;
  float* C;
  uint16_t* Cb;        // bf16 output, fp16 with cb_f16
  int cb_f16;
  int64_t ldc, ldcb;
  int accumulate;       // C += A . B^T instead of C = A . B^T (n_ks = 1)
  // device count (or null): c = *count - count_off.  kFwd/kGrad and count_axis
  // 0: rows r >= c are absent (not read, not written); count_axis 1 (kGemm):
  // the reduction stops at round_up(c, 128).  With both C and Cb, the output
  // is Cb = bf16(A . B^T (+ C when accumulate)) if *count <= final_at and C
  // otherwise; an empty reduction with accumulate set writes nothing.
  const int64_t* count;
  int64_t count_off;
  int count_axis;
  int64_t final_at;
};

template <int MODE, class E>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
void lce_tile_kernel(LceParams P) {
  using frag = typename Mma<E>::frag;
  using acc_t = typename Mma<E>::acc_t;
  constexpr int kT = Mma<E>::kT, kTM = kWM / kT, kTN = kWN / kT, kAV = kT * kT / kWave;
  constexpr int kKK = kRowBytes / (kWave / kT * 16);  // fragment steps (MFMA blocks) per stage
  static_assert(MODE == kGemm || sizeof(typename E::raw) == 2, "fp32 operands: plain GEMM only");
  constexpr int kES = (int)sizeof(typename E::raw);  // bytes per element
  constexpr int kSKE = kRowBytes / kES;              // hidden elements per stage
  // Two arrays rather than one, so that the compiler tracks the direct loads
  // into each stage on their own and an LDS read waits only for its stage.
  __shared__ __align__(1024) unsigned char st0[kStageBytes];
  __shared__ __align__(1024) unsigned char st1[kStageBytes];
  __shared__ int s_tcol[kBM];
  __shared__ float s_m[kBM], s_ls[kBM], s_g[kBM];
  auto stage_ptr = [&](int s) -> unsigned char* { return s == 0 ? st0 : st1; };

  // Tile order.  Workgroups are dispatched to the 8 XCDs round-robin
  // (XCD = blockIdx % 8) and each XCD has its own L2, so each XCD takes one
  // contiguous run of a grouped order (kGroupM row tiles sweep the vocabulary
  // together): the ~32 workgroups resident on an XCD then cover about
  // kGroupM row tiles x 4 column tiles and share their H and W reads in L2.
  // (A plain GEMM's hidden-dimension splits are the outermost index.)
  // A device count of rows shortens the row range; the tile order then covers
  // only the row tiles that hold rows (so every XCD keeps its share of the
  // work) and the workgroups past them return at once.
  int64_t row_end = P.row0 + P.nrows;
  int64_t k_end = P.Hd;
  bool to_bf16 = P.Cb != nullptr;
  if (P.count != nullptr) {
    const int64_t c = *P.count - P.count_off;
    if (MODE != kGemm || P.count_axis == 0) {
      if (c < row_end) row_end = c;
    } else {
      constexpr int64_t kstep = kStages * kSKE;
      const int64_t ke = c <= 0 ? 0 : (c + kstep - 1) / kstep * kstep;
      if (ke < k_end) k_end = ke;
      if (ke == 0 && P.accumulate) return;
      if (P.C != nullptr && P.Cb != nullptr) to_bf16 = *P.count <= P.final_at;
    }
  }
  row_end = uniform(row_end);
  k_end = uniform(k_end);
  if (row_end <= P.row0) return;
  const int64_t n_mt = (row_end - P.row0 + kBM - 1) / kBM;  // <= P.n_mt
  const int64_t tiles2 = n_mt * P.n_nt;
  const int64_t ntiles = tiles2 * (MODE == kGemm ? P.n_ks : 1);
  const int64_t per_xcd = (ntiles + kXcds - 1) / kXcds;
  // (the grid holds per_xcd workgroups per XCD only without a count)
  if ((int64_t)(blockIdx.x / kXcds) >= per_xcd) return;
  const int64_t gi0 = (int64_t)(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
  if (gi0 >= ntiles) return;
  const int64_t ks = uniform(gi0 / tiles2);
  const int64_t gi = gi0 - ks * tiles2;
  const int64_t per_group = (int64_t)kGroupM * P.n_nt;
  const int64_t group = gi / per_group;
  const int64_t first_m = group * kGroupM;
  const int64_t gsize = (n_mt - first_m < kGroupM) ? (n_mt - first_m) : kGroupM;
  const int64_t in_group = gi - group * per_group;
  // wave-uniform by construction; said so, or the compiler may keep the buffer
  // resources made from them in vector registers and loop over lanes at every load
  const int64_t mt = uniform(first_m + in_group % gsize);
  const int64_t nt = uniform(in_group / gsize);
  const int64_t m0 = P.row0 + mt * kBM;  // absolute first row
  const int64_t n0 = nt * kBN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  // per-row metadata of the tile (kThreads == kBM: one row per thread)
  float my_g = 0.f;
  if constexpr (MODE != kGemm) {
    const int64_t r = m0 + tid;
    int tc = -1;
    float lm = 0.f, ll = 0.f;
    if (r < row_end) {
      const int64_t s = r / P.bsz, b = r - s * P.bsz;
      const int64_t t = P.target[b * P.tsb + s * P.tss];
      const bool tmask = (t < P.vs) || (t >= P.ve) || (t - P.vs >= P.V);
      if (!tmask) {
        const int64_t c = t - P.vs - n0;
        if (c >= 0 && c < kBN) tc = (int)c;
      }
      if (MODE == kGrad) {
        my_g = P.g[b * P.gsb + s * P.gss];
        lm = P.stats[2 * r];
        ll = P.stats[2 * r + 1];
      }
    }
    s_tcol[tid] = tc;
    if (MODE == kGrad) {
      s_g[tid] = my_g;
      s_m[tid] = lm;
      s_ls[tid] = ll;
    }
  }
  if (MODE == kGrad) {
    // (onehot - p) * 0 == 0: a tile whose rows all have a zero upstream
    // gradient is written as zeros without the GEMM.
    if (!__syncthreads_or(my_g != 0.f)) {
      const int cvec = kBN / 8;
      for (int q = tid; q < kBM * cvec; q += kThreads) {
        const int rl = q / cvec, cv = q - rl * cvec;
        const int64_t r = m0 + rl;
        const int64_t c = n0 + cv * 8;
        if (r >= row_end || c >= P.V) continue;
        uint16_t* dst = P.G + (r - P.row0) * P.ldg + c;
        if (c + 8 <= P.V && ((reinterpret_cast<uintptr_t>(dst) & 15u) == 0)) {
          *reinterpret_cast<vu4*>(dst) = vu4{0u, 0u, 0u, 0u};
        } else {
          for (int e = 0; e < 8 && c + e < P.V; ++e) dst[e] = 0;
        }
      }
      if (P.Gt != nullptr && n0 + tid < P.V) {
        uint16_t* dt = P.Gt + (n0 + tid) * P.ldgt + (m0 - P.row0);
        for (int r8 = 0; r8 < kBM / 8; ++r8) *reinterpret_cast<vu4*>(dt + r8 * 8) = vu4{0u, 0u, 0u, 0u};
      }
      return;
    }
  }

  // ---- main loop: acc = H[m0 : m0+256] . W[n0 : n0+256]^T ----
  //
  // Direct loads go through buffer resources covering the tile's valid rows.
  // The row offset is in the VGPR offset, which the range check covers, so rows
  // past the end of H or W read as zero with no branch; the SGPR offset carries
  // only the stage's hidden offset, which stays inside a valid row.
  //
  // One direct load moves 8 rows x 128 B: lane l writes LDS bytes
  // [16 l, 16 l + 16) of the load's 1 KB block, i.e. row l / 8, slot l % 8, so
  // it fetches global chunk (l % 8) ^ ((row / 2) % 8) of that row (the inverse
  // of the lds_off swizzle).  Each wave issues kDmaPerWave loads of H and of W
  // per stage.
  // this tile's range of the hidden dimension (the whole of it but for split GEMMs)
  const int64_t kbase = (MODE == kGemm) ? ks * P.kb_len : 0;
  const int64_t krest = k_end - kbase < 0 ? 0 : k_end - kbase;
  const int64_t klen = (MODE == kGemm) ? (krest < P.kb_len ? krest : P.kb_len) : P.Hd;
  const int nst = (int)(klen / kSKE);  // a multiple of kStages (0: an empty reduction)
  if (MODE == kGemm && nst == 0) {
    // an empty reduction range (a reduction-length count, or a split past it):
    // the product is zero; handled here, before the accumulators exist
    for (int q = threadIdx.x; q < kBM * kBN; q += kThreads) {
      const int64_t row = m0 + q / kBN, col = n0 + q % kBN;
      if (row >= row_end || col >= P.V) continue;
      if (to_bf16) {
        const float o = (P.accumulate && P.C != nullptr) ? P.C[row * P.ldc + col] : 0.f;
        P.Cb[row * P.ldcb + col] = P.cb_f16 ? bits_of<F16>(o) : bits_of<BF16>(o);
      } else if (!P.accumulate) {
        P.C[(ks * P.nrows + row) * P.ldc + col] = 0.f;
      }
    }
    return;
  }
  const int64_t a_rows = (row_end - m0 < kBM) ? (row_end - m0) : kBM;
  const int64_t b_rows = (P.V - n0 < kBN) ? (P.V - n0) : kBN;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(static_cast<const char*>(P.h) + (m0 * P.ldh + kbase) * kES), 0,
      (int)((a_rows * P.ldh - kbase) * kES), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(static_cast<const char*>(P.w) + (n0 * P.ldw + kbase) * kES), 0,
      (int)((b_rows * P.ldw - kbase) * kES), 0x00020000);
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  int voff_a[kDmaPerWave], voff_b[kDmaPerWave];
#pragma unroll
  for (int i = 0; i < kDmaPerWave; ++i) {
    const int row = (wave * kDmaPerWave + i) * kDmaRows + (lane >> 3);
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    voff_a[i] = (int)(row * P.ldh * kES) + chunk * 16;
    voff_b[i] = (int)(row * P.ldw * kES) + chunk * 16;
  }
  // load q of stage data t: q < kDmaPerWave is an H block, else a W block
  auto dma = [&](unsigned char* stage, int t, int q) {
    const int soff = t * kRowBytes;
    if (q < kDmaPerWave) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc_a, (lds_ptr_t)(stage + (wave_u * kDmaPerWave + q) * kDmaBytes), 16, voff_a[q], soff, 0, 0);
    } else {
      const int qb = q - kDmaPerWave;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc_b, (lds_ptr_t)(stage + kHalfBytes + (wave_u * kDmaPerWave + qb) * kDmaBytes), 16,
          voff_b[qb], soff, 0, 0);
    }
  };

  // fragment read offsets: row (wm*128 | wn*128) + i*kT + lane % kT, the lane group's
  // chunk of step kk
  const int frow = lane & (kT - 1);
  int frag_off[kKK];
#pragma unroll
  for (int kk = 0; kk < kKK; ++kk) frag_off[kk] = lds_off(frow, kk * (kWave / kT) + lane / kT);
  frag fa[2][kTM], fb[2][kTN];
  // Reads go out in the order the MFMAs first need them: A0, all B, the other A (1% on
  // the forward against all A, all B).
  auto fread = [&](int set, const unsigned char* stage, int kk, int n) __attribute__((always_inline)) {
    // idx < kTM: A fragment idx; else B fragment idx - kTM
    const int idx = n == 0 ? 0 : n <= kTN ? kTM + n - 1 : n - kTN;
    if (idx < kTM)
      fa[set][idx] = *reinterpret_cast<const frag*>(stage + (wm * kWM + idx * kT) * kRowBytes + frag_off[kk]);
    else
      fb[set][idx - kTM] = *reinterpret_cast<const frag*>(
          stage + kHalfBytes + (wn * kWN + (idx - kTM) * kT) * kRowBytes + frag_off[kk]);
  };

  acc_t acc[kTM][kTN];
  auto clear_acc = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kTM; ++i)
#pragma unroll
      for (int j = 0; j < kTN; ++j)
#pragma unroll
        for (int v = 0; v < kAV; ++v) acc[i][j][v] = 0.f;
  };
  clear_acc();
  auto mfma = [&](int set, int q) __attribute__((always_inline)) {
    const int i = q / kTN, j = q % kTN;
    acc[i][j] = Mma<E>::run(fb[set][j], fa[set][i], acc[i][j]);
  };

  constexpr int kL = 2 * kDmaPerWave;  // direct loads per wave and stage
  constexpr int kMB = kTM * kTN;        // MFMAs per block
  constexpr int kReadEvery = kMB / (2 * (kTM + kTN)) > 1 ? 2 : 1, kLoadEvery = kMB / kL;
  static_assert(kKK % 2 == 0 && kLoadEvery * kL == kMB && kReadEvery * (kTM + kTN) <= kMB,
                "a block's reads and loads fit beside its MFMAs");
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  using T_ = std::integral_constant<bool, true>;
  using F_ = std::integral_constant<bool, false>;
  // One stage t (S = t % 2): kKK blocks of MFMAs (two of 64 for 16-bit operands, 32
  // hidden elements each).  While block kk runs on fragment set kk % 2, block kk + 1's
  // fragments are read into the other set.  Before the last block this wave waits for
  // its loads of stage data t + 1 (the only ones in flight) and the workgroup barrier
  // makes every wave's loads visible and ends every read of stage S (the last block's
  // fragments were read beside the block before).  The last block then reads the next
  // stage's block-0 fragments and issues the direct loads of stage data t + 2 into stage
  // S, spread over its MFMAs: 64 KB for the CU's LDS write port in half a stage.  (In a
  // quarter of the stage, forward 15.8 ms against 15.05, dW 6.42 against 5.88, dH 6.11
  // against 5.79 on [16384 | 5888, 4096] x [151808, 4096], all with 32 x 32 MFMAs; over
  // three quarters 15.57 ms: the last loads then come too late.)
  auto step = [&](int t, auto s_c, auto next_c, auto load_c) __attribute__((always_inline)) {
    constexpr int S = decltype(s_c)::value;
    constexpr bool NEXT = decltype(next_c)::value;
    constexpr bool LOAD = decltype(load_c)::value;
    unsigned char* cur = stage_ptr(S);
    const unsigned char* nxt = stage_ptr(S ^ 1);
#pragma unroll
    for (int kk = 0; kk < kKK - 1; ++kk) {
#pragma unroll
      for (int q = 0; q < kMB; ++q) {
        mfma(kk & 1, q);
        if (q % kReadEvery == 0 && q / kReadEvery < kTM + kTN) fread((kk + 1) & 1, cur, kk + 1, q / kReadEvery);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (NEXT) wait_vm_barrier<0>();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < kMB; ++q) {
      mfma(1, q);
      if constexpr (NEXT) {
        if (q % kReadEvery == 0 && q / kReadEvery < kTM + kTN) fread(0, nxt, 0, q / kReadEvery);
      }
      if constexpr (LOAD) {
        if (q % kLoadEvery == kLoadEvery / 4) dma(cur, t + 2, q / kLoadEvery);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto run_stages = [&]() __attribute__((always_inline)) {
    // Prologue: stage data 0 and 1 in flight; wait for 0 and read its block-0 fragments.
#pragma unroll
    for (int q = 0; q < kL; ++q) dma(st0, 0, q);
#pragma unroll
    for (int q = 0; q < kL; ++q) dma(st1, 1, q);
    wait_vm_barrier<kL>();
#pragma unroll
    for (int idx = 0; idx < kTM + kTN; ++idx) fread(0, st0, 0, idx);
    int t = 0;
    for (; t < nst - kStages; t += kStages) {
      step(t, S0{}, T_{}, T_{});
      step(t + 1, S1{}, T_{}, T_{});
    }
    step(t, S0{}, T_{}, F_{});
    step(t + 1, S1{}, F_{}, F_{});
  };

  float unscale = 1.f;  // what the accumulators are to be multiplied by (fp32 operands)
  if constexpr (std::is_same<E, F32>::value) {
    // ---- fp32 operands as three bf16 planes each ----
    //
    // x = x0 + x1 + x2 exactly, with x0 = bf16(x), x1 = bf16(x - x0) and
    // x2 = x - x0 - x1 (at most eight significant bits are left), so a product of
    // two elements is the sum of nine bf16 products; the three below 2^-25 of it
    // (a1 b2, a2 b1, a2 b2) are left out and the six others summed into the same
    // fp32 accumulators, the small ones first.  The fp32 MFMA runs at 1/16 of the bf16
    // rate, so six bf16 products cost 3/8 of one fp32 product, and 32 k-terms enter an
    // accumulator in 12 roundings instead of 16: [2048, 4096] x [65536, 4096]^T 151 -> 241
    // TFLOP/s back to back (1450 of bf16), error against 64 bits 1.15e-6 -> 1.00e-6 of the root
    // of the sum of squared products (K = 64: 1.44e-7 -> 1.10e-7; sums of two terms 3.1e-8
    // -> 3.3e-8, of one 2.5e-8 -> 3.4e-8: what is left out counts there).  Bound by the MFMA
    // units, busy 87% of the cycles at the 1.5 GHz that this load leaves (82% at 1.92 GHz
    // and 276 TFLOP/s where memory-bound kernels run in between).
    //
    // Unscaled, the planes hold all of x from 2^-109 on, and the logits gradient (the
    // first operand of dH and dW) is less for every improbable token: one such value
    // sends its tile through both loops below.  So the first operand is multiplied by
    // 2^40 before it is split and the result by 2^-40: its planes then hold every x below
    // 2^88, subnormal ones too.  Step of [1024, 2, 4096] x [151936, 4096], every row
    // active: with logits of standard deviation 10 83.1 -> 50.5 ms, of 1.5 49.4 and 49.3.
    // (Both operands by 2^24, without the check of the residuals, takes 3% more.)
    //
    // Each lane reads the fp32 fragments of the coming 16 hidden elements and
    // splits them while the 96 MFMAs of the current ones run: 56 VALU
    // instructions per fragment (second operand 48), five or six in the shadow of each
    // MFMA.  (Residuals by v_dot2_f32_bf16, 28 instructions, were slower: 207 TFLOP/s.)
    using frag16 = typename Mma<BF16>::frag;
    constexpr float kScale = 0x1p40f, kUnscale = 0x1p-40f;
    constexpr int kPl = 3, kFr = kTM + kTN;
    constexpr int kOpSlots = 11;  // slots a fragment's split takes
    constexpr int kSlots = 2 * kPl * kMB;            // MFMAs per 16 hidden elements
    constexpr int kOps = 52, kPer = 5;               // steps of a fragment's split, per slot
    constexpr int kFirst = kSlots - kFr * kOpSlots;  // slot of the first split op
    static_assert(kFirst >= 4 && kKK == 4, "reads ahead of the split");
    // the lane's 8 hidden elements 16 kk + 8 (lane / 32) + 0..7 of a row: two chunks
    int foff[2][2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int c = 0; c < 2; ++c) foff[kk][c] = lds_off(frow, kk * 4 + (lane >> 5) * 2 + c);
    frag16 pl[2][kFr][kPl];  // [set][A fragments, then B][plane]
    float raw[3][8];
    float h0, h1, r0, r1;
    uint32_t lost = 0;  // the third planes are the last residuals unless one has bits in its low half
    uint32_t out[kPl][4];
    auto read_raw = [&](const unsigned char* stage, int kk, int f) __attribute__((always_inline)) {
      const unsigned char* rows = f < kTM ? stage + (wm * kWM + f * 32) * kRowBytes
                                          : stage + kHalfBytes + (wn * kWN + (f - kTM) * 32) * kRowBytes;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const frag q = *reinterpret_cast<const frag*>(rows + foff[kk][c]);
#pragma unroll
        for (int e = 0; e < 4; ++e) raw[f % 3][c * 4 + e] = q[e];
      }
    };
    // op N of the split of fragment F into set SET
    auto split_op = [&](auto set_c, auto f_c, auto n_c) __attribute__((always_inline)) {
      constexpr int F = decltype(f_c)::value, N = decltype(n_c)::value;
      constexpr int P = N / 13, O = N % 13;
      float* x = raw[F % 3];
      if constexpr (O == 0) {
        if constexpr (F < kTM) {
          x[2 * P] *= kScale;
          x[2 * P + 1] *= kScale;
        }
      } else if constexpr (O == 1) out[0][P] = BF16::pack2(x[2 * P], x[2 * P + 1]);
      else if constexpr (O == 2) h0 = low_bf16(out[0][P]);
      else if constexpr (O == 3) h1 = __uint_as_float(out[0][P] & 0xffff0000u);
      else if constexpr (O == 4) r0 = x[2 * P] - h0;
      else if constexpr (O == 5) r1 = x[2 * P + 1] - h1;
      else if constexpr (O == 6) out[1][P] = BF16::pack2(r0, r1);
      else if constexpr (O == 7) h0 = low_bf16(out[1][P]);
      else if constexpr (O == 8) h1 = __uint_as_float(out[1][P] & 0xffff0000u);
      else if constexpr (O == 9) r0 = r0 - h0;
      else if constexpr (O == 10) r1 = r1 - h1;
      else if constexpr (O == 11) out[2][P] = BF16::pack2(r0, r1);
      else lost = or3(lost, r0, r1);
      if constexpr (N == kOps - 1) {
#pragma unroll
        for (int k = 0; k < kPl; ++k) {
          const vu4 q = {out[k][0], out[k][1], out[k][2], out[k][3]};
          pl[decltype(set_c)::value][F][k] = __builtin_bit_cast(frag16, q);
        }
      }
    };
    // One step: the 96 MFMAs of set SET (products a2 b0, a0 b2, a1 b1, a1 b0, a0 b1,
    // a0 b0 of the 16 tiles), beside them the reads and the split of the next 16
    // hidden elements (half kk of `stage`) into the other set, and with LOAD the
    // direct loads of stage data t_load into `into`.
    auto step16 = [&](auto set_c, const unsigned char* stage, int kk, auto load_c, unsigned char* into,
                      int t_load) __attribute__((always_inline)) {
      constexpr int SET = decltype(set_c)::value;
      constexpr bool LOAD = decltype(load_c)::value;
      static_for<kSlots>([&](auto q_c) __attribute__((always_inline)) {
        constexpr int Q = decltype(q_c)::value;
        constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
        constexpr int PR = Q / kMB, I = Q / kTN % kTM, J = Q % kTN;
        acc[I][J] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pl[SET][kTM + J][pb[PR]], pl[SET][I][pa[PR]],
                                                            acc[I][J], 0, 0, 0);
        // the first two fragments are read at once, each other one a split ahead
        if constexpr (Q == 0) read_raw(stage, kk, 0);
        if constexpr (Q == 2) read_raw(stage, kk, 1);
        if constexpr (Q >= kFirst) {
          constexpr int F = (Q - kFirst) / kOpSlots, N = (Q - kFirst) % kOpSlots * kPer;
          if constexpr (N == 0 && F + 2 < kFr) read_raw(stage, kk, F + 2);
          static_for<kPer>([&](auto u_c) __attribute__((always_inline)) {
            if constexpr (N + decltype(u_c)::value < kOps)
              split_op(std::integral_constant<int, SET ^ 1>{}, std::integral_constant<int, F>{},
                       std::integral_constant<int, N + decltype(u_c)::value>{});
          });
        }
        if constexpr (LOAD && Q % 4 == 1 && Q / 4 < kL) dma(into, t_load, Q / 4);
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    // Prologue: stage data 0 and 1 in flight, the first 16 elements split.
#pragma unroll
    for (int q = 0; q < kL; ++q) dma(st0, 0, q);
#pragma unroll
    for (int q = 0; q < kL; ++q) dma(st1, 1, q);
    wait_vm_barrier<kL>();
    static_for<kFr>([&](auto f_c) __attribute__((always_inline)) {
      read_raw(st0, 0, decltype(f_c)::value);
      static_for<kOps>([&](auto n_c) __attribute__((always_inline)) { split_op(S0{}, f_c, n_c); });
    });
    // Stage t: step 0 computes its first half and splits its second; then every
    // wave has read the stage and, past the barrier, step 1 refills it with stage
    // data t + 2 while it splits the first half of stage t + 1.  Past the last
    // stage the loads and the split repeat the last stage's data, unused.
    auto stage2 = [&](int t, auto s_c) __attribute__((always_inline)) {
      constexpr int S = decltype(s_c)::value;
      unsigned char* cur = stage_ptr(S);
      step16(S0{}, cur, 1, F_{}, cur, 0);
      wait_vm_barrier<0>();
      step16(S1{}, stage_ptr(S ^ 1), 0, T_{}, cur, t + 2 < nst ? t + 2 : nst - 1);
    };
    for (int t = 0; t < nst; t += kStages) {
      stage2(t, S0{});
      stage2(t + 1, S1{});
    }
    wait_vm_barrier<0>();
    // Infinities and NaN do not split (inf - inf), nor does a value that the scale
    // takes to infinity or that rounds there as a bf16; a sum of 2^88 overflows under
    // the scale; and a second operand below 2^-109 can have bits that its planes do not
    // hold: a tile in which one shows is formed again with fp32 MFMAs.
    float z = 0.f;
#pragma unroll
    for (int i = 0; i < kTM; ++i)
#pragma unroll
      for (int j = 0; j < kTN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) z += acc[i][j][v] * 0.f;
    unscale = kUnscale;
    if (__syncthreads_or(!(z == 0.f) || (lost & 0xffffu) != 0)) {
      clear_acc();
      run_stages();
      unscale = 1.f;
    }
  } else {
    run_stages();
  }

  if constexpr (MODE == kGemm) {
    // ---- plain GEMM: the accumulators go straight to C ----
    // a 16-bit output over an fp32 running sum adds C before it rounds
    const bool add_c = P.accumulate && P.C != nullptr;
    float* C = P.C == nullptr ? nullptr : P.C + ks * P.nrows * P.ldc;
    // each lane holds groups of four consecutive columns of a row, moved as one
    // 16-byte (fp32) or 8-byte (16-bit) piece where base and row stride allow.  One
    // unrolled loop per kind of store: a single loop choosing its store per element
    // grew past what the compiler unrolls and put the accumulators on the stack.
    const bool vec_c = C != nullptr && (reinterpret_cast<uintptr_t>(C) & 15u) == 0 && P.ldc % 4 == 0;
    const bool vec_b = P.Cb != nullptr && (reinterpret_cast<uintptr_t>(P.Cb) & 7u) == 0 && P.ldcb % 4 == 0;
    auto each = [&](auto&& put) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < kTM; ++i) {
        const int64_t row = m0 + wm * kWM + i * kT + frow;
        if (row >= row_end) continue;
#pragma unroll
        for (int j = 0; j < kTN; ++j)
#pragma unroll
          for (int g = 0; g < kAV / 4; ++g) {
            const int64_t col = n0 + wn * kWN + j * kT + g * 8 + lane / kT * 4;
            f32x4 o = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
            if constexpr (std::is_same<E, F32>::value) {
#pragma unroll
              for (int e = 0; e < 4; ++e) o[e] *= unscale;
            }
            if (col < P.V) put(row, col, o, col + 4 <= P.V);
          }
      }
    };
    auto load_c = [&](int64_t row, int64_t col, bool full) {
      const float* src = C + row * P.ldc + col;
      f32x4 c = {0.f, 0.f, 0.f, 0.f};
      if (full && vec_c) {
        c = *reinterpret_cast<const f32x4*>(src);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < P.V) c[e] = src[e];
      }
      return c;
    };
    auto store_c = [&](int64_t row, int64_t col, f32x4 o, bool full) {
      float* dst = C + row * P.ldc + col;
      if (full && vec_c) {
        *reinterpret_cast<f32x4*>(dst) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < P.V) dst[e] = o[e];
      }
    };
    auto store_b = [&](auto eb, int64_t row, int64_t col, f32x4 o, bool full) {
      using EB = decltype(eb);
      uint16_t* dst = P.Cb + row * P.ldcb + col;
      const uint2 w = pack4<EB>(o);
      if (full && vec_b) {
        *reinterpret_cast<uint2*>(dst) = w;
      } else {
        const uint32_t wv[2] = {w.x, w.y};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < P.V) dst[e] = (uint16_t)(wv[e >> 1] >> (16 * (e & 1)));
      }
    };
    auto out_b = [&](auto eb) __attribute__((always_inline)) {
      if (add_c)
        each([&](int64_t row, int64_t col, f32x4 o, bool full)
                 __attribute__((always_inline)) { store_b(eb, row, col, load_c(row, col, full) + o, full); });
      else
        each([&](int64_t row, int64_t col, f32x4 o, bool full)
                 __attribute__((always_inline)) { store_b(eb, row, col, o, full); });
    };
    constexpr bool k16 = !std::is_same<E, F32>::value;  // 16-bit outputs: 16-bit operands only
    if (k16 && to_bf16 && P.cb_f16) {
      if constexpr (k16) out_b(F16{});
    } else if (k16 && to_bf16) {
      if constexpr (k16) out_b(BF16{});
    } else if (add_c)
      each([&](int64_t row, int64_t col, f32x4 o, bool full)
               __attribute__((always_inline)) { store_c(row, col, load_c(row, col, full) + o, full); });
    else
      each([&](int64_t row, int64_t col, f32x4 o, bool full)
               __attribute__((always_inline)) { store_c(row, col, o, full); });
  } else {
  // ---- epilogue: the tile goes through LDS as bf16, one row per thread ----
  //
  // The accumulators of a row are spread over lanes and waves; instead of cross-lane
  // reductions each wave writes its quarter to LDS (row-major [256][256] bf16
  // over the two stage arrays, 16-byte chunks XOR-swizzled by row; each lane
  // four consecutive columns of a row at a time) and thread t then walks row t
  // (forward) or copies rows out with 16-byte stores (gradient).  Every direct load
  // has landed (the last wait was vmcnt(0)); the barrier orders every wave's last
  // fragment reads before the stores.
  wait_vm_barrier<0>();
  const int wm_u = wave_u >> 1;
  const int col_lane = (lane >> 4) * 4;  // the lane's first column of an MFMA tile
  // the epilogue rows of this wave's quarter live in stage array wm
  uint16_t* const xq = reinterpret_cast<uint16_t*>(stage_ptr(wm_u));
  if (MODE == kFwd) {
#pragma unroll
    for (int i = 0; i < kTM; ++i) {
      const int rl = wm * kWM + i * kT + frow;
#pragma unroll
      for (int j = 0; j < kTN; ++j)
        *reinterpret_cast<uint2*>(xq + xs_index(rl, wn * kWN + j * kT + col_lane)) = pack4<E>(acc[i][j]);
    }
    __syncthreads();
    const int64_t r = m0 + tid;
    if (r < row_end) {
      // row tid is local row tid % 128 of stage array tid / 128
      const uint16_t* xs = reinterpret_cast<const uint16_t*>(stage_ptr(wm_u));
      const int ncols = (P.V - n0 < kBN) ? (int)(P.V - n0) : kBN;
      const vu4* rowp = reinterpret_cast<const vu4*>(xs + (tid & (kEpiRows - 1)) * kBN);
      const int sw = xs_swizzle(tid);
      float M = -INFINITY, sum = 0.f;
      // two passes (max, then sum of exp); the column bound is only checked in
      // the last, partial column tile
      auto walk = [&](auto full_c) {
        constexpr bool FULL = decltype(full_c)::value;
        for (int c = 0; c < kBN / 8; ++c) {
          float w[8];
          E::unpack(rowp[c ^ sw], w);
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (FULL || c * 8 + e < ncols) M = fmaxf(M, w[e]);
        }
        if (M != -INFINITY) {
          float s4[4] = {0.f, 0.f, 0.f, 0.f};
          for (int c = 0; c < kBN / 8; ++c) {
            float w[8];
            E::unpack(rowp[c ^ sw], w);
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (FULL || c * 8 + e < ncols) s4[e & 3] += fast_exp2((w[e] - M) * kLog2e);
          }
          sum = (s4[0] + s4[1]) + (s4[2] + s4[3]);
        }
      };
      if (ncols == kBN)
        walk(std::true_type{});
      else
        walk(std::false_type{});
      float* dst = P.part + ((r - P.row0) * P.n_nt + nt) * 2;
      dst[0] = M;
      dst[1] = sum;
      const int tc = s_tcol[tid];
      if (tc >= 0) P.xt[r - P.row0] = value_of<E>(xs[xs_index(tid, tc)]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < kTM; ++i) {
      const int rl = wm * kWM + i * kT + frow;
      const float gv = s_g[rl], M = s_m[rl], LS = s_ls[rl];
      const int tc = s_tcol[rl];
#pragma unroll
      for (int j = 0; j < kTN; ++j) {
        const int cl = wn * kWN + j * kT + col_lane;
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          float x0 = acc[i][j][e], x1 = acc[i][j][e + 1];
          round_trip2<E>(x0, x1);  // the logits in the operand dtype
          o[e] = fast_exp2(((x0 - M) - LS) * kLog2e);
          o[e + 1] = fast_exp2(((x1 - M) - LS) * kLog2e);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (cl + e == tc) ? (1.f - o[e]) * gv : -o[e] * gv;
        // G is bf16 for either operand dtype
        *reinterpret_cast<uint2*>(xq + xs_index(rl, cl)) = pack4<BF16>(o);
      }
    }
    __syncthreads();
    // 32 threads per row, one 16-byte chunk each; 8 rows per pass
    const int c = tid & 31;
#pragma unroll 4
    for (int k = 0; k < kBM / 8; ++k) {
      const int rl = (tid >> 5) + 8 * k;
      const int64_t r = m0 + rl;
      const int64_t col0 = n0 + c * 8;
      if (r >= row_end || col0 >= P.V) continue;
      const uint16_t* xs = reinterpret_cast<const uint16_t*>(stage_ptr(rl / kEpiRows));
      const vu4 q = reinterpret_cast<const vu4*>(xs + (rl & (kEpiRows - 1)) * kBN)[c ^ xs_swizzle(rl)];
      uint16_t* dst = P.G + (r - P.row0) * P.ldg + col0;
      if (col0 + 8 <= P.V && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
        *reinterpret_cast<vu4*>(dst) = q;
      } else {
        const uint32_t wv[4] = {q.x, q.y, q.z, q.w};
        for (int e = 0; e < 8 && col0 + e < P.V; ++e)
          dst[e] = (uint16_t)(wv[e >> 1] >> ((e & 1) * 16));
      }
    }
    if (P.Gt != nullptr) {
      // the transposed tile (rows of G past its end are zeros, which the caller's
      // padded reduction length relies on): a wave takes 16 columns x 64 rows at a time,
      // lane l the column pair l % 8 and the eight rows from 8 (l / 8) on, so that eight
      // lanes store one 128-byte line of G^T (one column per lane, 64 lines open per
      // store, took 0.6-0.7 ms of 6.8 on [5888, 4096] x [151808, 4096]; this takes 0.3 of 6.1)
#pragma unroll 2
      for (int it = 0; it < kBN / 16 * (kBM / 64) / kWaves; ++it) {
        const int q = wave_u * (kBN / 16 * (kBM / 64) / kWaves) + it;
        const int cl = (q % (kBN / 16)) * 16 + (lane & 7) * 2;
        const int rl = (q / (kBN / 16)) * 64 + (lane >> 3) * 8;
        const int64_t col = n0 + cl;
        if (col >= P.V) continue;
        const uint16_t* xs = reinterpret_cast<const uint16_t*>(stage_ptr(rl / kEpiRows));
        uint16_t* dst = P.Gt + col * P.ldgt + (m0 - P.row0) + rl;
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // two rows' pairs of columns -> two columns' pairs of rows
          const uint32_t a = *reinterpret_cast<const uint32_t*>(xs + xs_index(rl + 2 * e, cl));
          const uint32_t b = *reinterpret_cast<const uint32_t*>(xs + xs_index(rl + 2 * e + 1, cl));
          lo[e] = (a & 0xffffu) | (b << 16);
          hi[e] = (a >> 16) | (b & 0xffff0000u);
        }
        *reinterpret_cast<vu4*>(dst) = vu4{lo[0], lo[1], lo[2], lo[3]};
        if (col + 1 < P.V) *reinterpret_cast<vu4*>(dst + P.ldgt) = vu4{hi[0], hi[1], hi[2], hi[3]};
      }
    }
  }
  }  // the fused epilogues
}

// dst[c][r] = bf16(src[r][c]) for r < R, c < C, and dst[c][r] = 0 for
// R <= r < Rp (src of dtype ES, bf16 or fp16; dst rows of stride ldd >= Rp),
// R = min(R, *count) when count is given.  64 x 64 tiles through LDS, moved
// as 16-byte pieces (eight elements of a row in, eight of a column out) where
// the pointers, strides and tile edges allow, element by element elsewhere.
template <class ES>
__global__ __launch_bounds__(256) void transpose_bf16_kernel(const uint16_t* __restrict__ src,
                                                             int64_t R, int64_t C, int64_t lds,
                                                             uint16_t* __restrict__ dst,
                                                             int64_t ldd, int64_t Rp,
                                                             int64_t n_ct,
                                                             const int64_t* __restrict__ count) {
  // row pitch 66 elements (33 words): the eight rows 8 apart that a wave's
  // column reads touch start in different LDS banks
  constexpr int kP = 66;
  __shared__ uint16_t tile[64 * kP];
  if (count != nullptr && *count < R) R = *count;
  const int64_t tr = blockIdx.x / n_ct, tc = blockIdx.x - tr * n_ct;
  const int64_t r0 = tr * 64, c0 = tc * 64;
  const bool vin = ((lds & 7) | (reinterpret_cast<uintptr_t>(src) & 15)) == 0;
  const bool vout = ((ldd & 7) | (reinterpret_cast<uintptr_t>(dst) & 15)) == 0;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int idx = (int)threadIdx.x + 256 * k, lr = idx >> 3, cg = (idx & 7) * 8;
    const int64_t r = r0 + lr, c = c0 + cg;
    uint32_t w[4];
    if (vin && r < R && c + 8 <= C) {
      const vu4 q = *reinterpret_cast<const vu4*>(src + r * lds + c);
      w[0] = q.x; w[1] = q.y; w[2] = q.z; w[3] = q.w;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t lo = (r < R && c + 2 * j < C) ? src[r * lds + c + 2 * j] : 0u;
        const uint32_t hi = (r < R && c + 2 * j + 1 < C) ? src[r * lds + c + 2 * j + 1] : 0u;
        w[j] = lo | (hi << 16);
      }
    }
    if constexpr (std::is_same<ES, F16>::value) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        w[j] = (uint32_t)bits_of<BF16>(value_of<F16>((uint16_t)(w[j] & 0xffffu))) |
               ((uint32_t)bits_of<BF16>(value_of<F16>((uint16_t)(w[j] >> 16))) << 16);
    }
    // (lr * 66 + cg) elements = a whole number of 4-byte words
    uint32_t* t32 = reinterpret_cast<uint32_t*>(tile + lr * kP + cg);
#pragma unroll
    for (int j = 0; j < 4; ++j) t32[j] = w[j];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int idx = (int)threadIdx.x + 256 * k, lc = idx >> 3, rg = (idx & 7) * 8;
    const int64_t c = c0 + lc, r = r0 + rg;
    if (c >= C) continue;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = (uint32_t)tile[(rg + 2 * j) * kP + lc] | ((uint32_t)tile[(rg + 2 * j + 1) * kP + lc] << 16);
    uint16_t* d = dst + c * ldd + r;
    if (vout && r + 8 <= Rp) {
      *reinterpret_cast<vu4*>(d) = vu4{w[0], w[1], w[2], w[3]};
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (r + i < Rp) d[i] = (uint16_t)(w[i >> 1] >> (16 * (i & 1)));
    }
  }
}

// dst[c][r] = src[r][c] for r < R, c < C, and dst[c][r] = 0 for R <= r < Rp
// (fp32; dst rows of stride ldd >= Rp), R = min(R, *count - count_off) when
// count is given.  64 x 64 tiles through LDS, moved as 16-byte pieces (four
// elements of a row in, four of a column out) where the pointers, strides and
// tile edges allow, element by element elsewhere.
__global__ __launch_bounds__(256) void transpose_f32_kernel(const float* __restrict__ src, int64_t R,
                                                            int64_t C, int64_t lds,
                                                            float* __restrict__ dst, int64_t ldd,
                                                            int64_t Rp, int64_t n_ct,
                                                            const int64_t* __restrict__ count,
                                                            int64_t count_off) {
  // row pitch 65 words: a wave's row pieces and column reads each fall in
  // distinct LDS banks
  constexpr int kP = 65;
  __shared__ float tile[64 * kP];
  if (count != nullptr) {
    const int64_t c = *count - count_off;
    if (c < R) R = c < 0 ? 0 : c;
  }
  const int64_t tr = blockIdx.x / n_ct, tc = blockIdx.x - tr * n_ct;
  const int64_t r0 = tr * 64, c0 = tc * 64;
  const bool vin = ((lds & 3) | (reinterpret_cast<uintptr_t>(src) & 15)) == 0;
  const bool vout = ((ldd & 3) | (reinterpret_cast<uintptr_t>(dst) & 15)) == 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int idx = (int)threadIdx.x + 256 * k, lr = idx >> 4, cg = (idx & 15) * 4;
    const int64_t r = r0 + lr, c = c0 + cg;
    float w[4];
    if (vin && r < R && c + 4 <= C) {
      const float4 q = *reinterpret_cast<const float4*>(src + r * lds + c);
      w[0] = q.x; w[1] = q.y; w[2] = q.z; w[3] = q.w;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = (r < R && c + j < C) ? src[r * lds + c + j] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) tile[lr * kP + cg + j] = w[j];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int idx = (int)threadIdx.x + 256 * k, lc = idx >> 4, rg = (idx & 15) * 4;
    const int64_t c = c0 + lc, r = r0 + rg;
    if (c >= C) continue;
    float w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = tile[(rg + i) * kP + lc];
    float* d = dst + c * ldd + r;
    if (vout && r + 4 <= Rp) {
      *reinterpret_cast<float4*>(d) = make_float4(w[0], w[1], w[2], w[3]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (r + i < Rp) d[i] = w[i];
    }
  }
}

// out[r(m)][n] = EO(sum over s of part[s][m][n]) (EO bf16, fp16 or fp32), summed in split order,
// with r(m) = out_rows[m] when a row map is given (rows mapped outside
// [0, out_nrows) are skipped) and m otherwise; with a count, rows
// m >= *count - count_off are written as zeros without reading.  VEC
// consecutive elements per thread (N and ld multiples of VEC).
template <int VEC, class EO>
__global__ __launch_bounds__(256) void sum_splits_kernel(const float* __restrict__ part,
                                                         int64_t n_ks, int64_t M, int64_t N,
                                                         int64_t ld, void* __restrict__ out,
                                                         int64_t ldo,
                                                         const int64_t* __restrict__ out_rows,
                                                         int64_t out_nrows,
                                                         const int64_t* __restrict__ count,
                                                         int64_t count_off) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * VEC;
  if (i >= M * N) return;
  const int64_t m = i / N, n = i - m * N;
  int64_t r = m;
  if (out_rows != nullptr) {
    r = out_rows[m];
    if (r < 0 || r >= out_nrows) return;
  }
  float acc[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) acc[e] = 0.f;
  if (count == nullptr || m < *count - count_off) {
    for (int64_t s = 0; s < n_ks; ++s) {
      const float* src = part + (s * M + m) * ld + n;
      if constexpr (VEC == 4) {
        const float4 q = *reinterpret_cast<const float4*>(src);
        acc[0] += q.x;
        acc[1] += q.y;
        acc[2] += q.z;
        acc[3] += q.w;
      } else {
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] += src[e];
      }
    }
  }
  if constexpr (std::is_same<EO, F32>::value) {
    float* dst = static_cast<float*>(out) + r * ldo + n;
    if constexpr (VEC == 4) {
      *reinterpret_cast<float4*>(dst) = float4{acc[0], acc[1], acc[2], acc[3]};
    } else {
#pragma unroll
      for (int e = 0; e < VEC; ++e) dst[e] = acc[e];
    }
  } else {
    uint16_t* dst = static_cast<uint16_t*>(out) + r * ldo + n;
    if constexpr (VEC == 4) {
      const uint32_t lo = (uint32_t)bits_of<EO>(acc[0]) | ((uint32_t)bits_of<EO>(acc[1]) << 16);
      const uint32_t hi = (uint32_t)bits_of<EO>(acc[2]) | ((uint32_t)bits_of<EO>(acc[3]) << 16);
      *reinterpret_cast<uint2*>(dst) = uint2{lo, hi};
    } else {
#pragma unroll
      for (int e = 0; e < VEC; ++e) dst[e] = bits_of<EO>(acc[e]);
    }
  }
}

// The rows r = (s, b) = (r / bsz, r % bsz) whose upstream gradient is not zero, in
// order, then the others from the end backwards: perm, the rows' gradients and the
// count of the first kind.  One workgroup, 8 x 1024 rows a step (their loads in
// flight together, a ballot and a sum over 16 waves per 1024).  With the gather below
// it takes the place of a stable sort, a sum and six gathers of the library: step of
// 137 rows x [1355, 4096] fp16 356 -> 248 us (host-bound), of 115 rows x [11749, 4096]
// bf16 441 -> 337; nothing to see at 16384 rows.
constexpr int kActThreads = 1024;
__global__ __launch_bounds__(kActThreads) void lce_active_rows_kernel(
    const float* __restrict__ g, int64_t gsb, int64_t gss, uint32_t T, uint32_t bsz,
    int64_t* __restrict__ perm, float* __restrict__ g_a, int64_t* __restrict__ count) {
  constexpr int NW = kActThreads / kWave, U = 8;
  __shared__ uint32_t wsum[2][NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t base = 0;  // active rows before this step
  for (uint32_t r0 = 0; r0 < T; r0 += U * kActThreads) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t r = r0 + u * kActThreads + tid;
      const uint32_t s = r / bsz, b = r - s * bsz;
      v[u] = r < T ? g[(int64_t)b * gsb + (int64_t)s * gss] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t r = r0 + u * kActThreads + tid;
      const bool act = r < T && v[u] != 0.f;
      const uint64_t bal = __ballot(act);
      // the two buffers alternate, so one barrier a round separates a round's
      // writes from the reads of the round before last
      if (lane == 0) wsum[u & 1][wave] = (uint32_t)__popcll(bal);
      __syncthreads();
      uint32_t before = base + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const uint32_t n = wsum[u & 1][w];
        before += w < wave ? n : 0u;
        base += n;
      }
      if (r < T) {
        const uint32_t at = act ? before : T - 1 - (r - before);
        perm[at] = r;
        g_a[at] = v[u];
      }
    }
  }
  if (tid == 0) *count = base;
}

// Row m of the permuted targets and statistics and, for m < *count, of the permuted
// hidden states (row_units units of UNIT per row; rows past the count stay as they
// are: every kernel stops at the count).  One workgroup per row, up to kGatherGrid of
// them: a launch holds fewer than 2^32 threads.
constexpr int64_t kGatherGrid = int64_t(1) << 20;
template <class UNIT>
__global__ __launch_bounds__(256) void lce_gather_rows_kernel(
    const int64_t* __restrict__ perm, const int64_t* __restrict__ count, int64_t T, uint32_t bsz,
    const int64_t* __restrict__ target, int64_t tsb, int64_t tss, const float* __restrict__ stats,
    const UNIT* __restrict__ hidden, int64_t row_units, int64_t ld_units, int64_t* __restrict__ tgt_a,
    float* __restrict__ st_a, UNIT* __restrict__ h_a) {
  for (int64_t m = blockIdx.x; m < T; m += kGatherGrid) {
    const uint32_t r = (uint32_t)perm[m];
    const bool live = m < *count;
    if (threadIdx.x == 0) {
      const uint32_t s = r / bsz, b = r - s * bsz;
      tgt_a[m] = target[(int64_t)b * tsb + (int64_t)s * tss];
      st_a[2 * m] = stats[2 * (int64_t)r];
      st_a[2 * m + 1] = stats[2 * (int64_t)r + 1];
    }
    if (!live) continue;
    const UNIT* src = hidden + (int64_t)r * ld_units;
    UNIT* dst = h_a + m * row_units;
    for (int64_t k = threadIdx.x; k < row_units; k += 256) dst[k] = src[k];
  }
}

// Per row: combine the column-tile partials into the row's max and log-sum-exp,
// then logprob = (x_t - max) - logsum (0 for targets outside the slice).
// One wave per row.
__global__ __launch_bounds__(256) void lce_merge_kernel(
    const float* __restrict__ part, const float* __restrict__ xt, int64_t row0, int64_t nrows,
    int64_t n_nt, int64_t bsz, const int64_t* __restrict__ target, int64_t tsb, int64_t tss,
    int64_t vs, int64_t ve, int64_t V, float* __restrict__ out, int64_t osb, int64_t oss,
    float* __restrict__ stats) {
  const int lane = threadIdx.x & 63;
  const int64_t rl = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (rl >= nrows) return;
  const float* p = part + rl * n_nt * 2;
  float M = -INFINITY;
  for (int64_t j = lane; j < n_nt; j += 64) M = fmaxf(M, p[2 * j]);
  M = wave_max(M);
  float s = 0.f;
  if (M != -INFINITY) {
    for (int64_t j = lane; j < n_nt; j += 64) {
      const float mj = p[2 * j];
      if (mj != -INFINITY) s += p[2 * j + 1] * fast_exp2((mj - M) * kLog2e);
    }
  }
  s = wave_sum(s);
  if (lane == 0) {
    const int64_t r = row0 + rl;
    const int64_t sq = r / bsz, b = r - sq * bsz;
    const int64_t t = target[b * tsb + sq * tss];
    const bool tmask = (t < vs) || (t >= ve) || (t - vs >= V);
    const float logsum = logf(s);
    out[b * osb + sq * oss] = tmask ? 0.f : (xt[rl] - M) - logsum;
    if (stats != nullptr) {
      stats[2 * r] = M;
      stats[2 * r + 1] = logsum;
    }
  }
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

int check_common(const void* hidden, int64_t T, int64_t Hd, int64_t ldh, const void* weight,
                 int64_t V, int64_t ldw, const int64_t* target, int64_t bsz) {
  MIRL_REQUIRE(hidden && weight && target, "null pointer argument");
  MIRL_REQUIRE(T >= 0 && V > 0 && Hd > 0 && bsz > 0, "invalid shape T=%lld V=%lld H=%lld B=%lld",
               (long long)T, (long long)V, (long long)Hd, (long long)bsz);
  MIRL_REQUIRE(T % bsz == 0, "row count %lld is not a multiple of the batch size %lld",
               (long long)T, (long long)bsz);
  MIRL_REQUIRE(Hd % (kStages * kSK) == 0, "hidden size %lld must be a multiple of %d", (long long)Hd,
               kStages * kSK);
  MIRL_REQUIRE(ldh < (int64_t(1) << 22) && ldw < (int64_t(1) << 22),
               "row strides (%lld, %lld) must be below 2^22 elements", (long long)ldh, (long long)ldw);
  MIRL_REQUIRE(ldh % 8 == 0 && ldw % 8 == 0 && ldh >= Hd && ldw >= Hd,
               "row strides (%lld, %lld) must be multiples of 8 elements and >= the hidden size",
               (long long)ldh, (long long)ldw);
  MIRL_REQUIRE((reinterpret_cast<uintptr_t>(hidden) & 15u) == 0 &&
                   (reinterpret_cast<uintptr_t>(weight) & 15u) == 0,
               "hidden states and weight must be 16-byte aligned");
  MIRL_REQUIRE(V < (int64_t(1) << 31) && T < (int64_t(1) << 31), "sizes exceed 2^31-1");
  return MIRL_OK;
}

}  // namespace
}  // namespace mirl

using namespace mirl;

extern "C" int64_t mirl_linear_ce_workspace_elems(int64_t T, int64_t V) {
  if (T <= 0 || V <= 0) return 0;
  return T * ceil_div(V, kBN) * 2 + T;
}

static bool lce_dtype_ok(int dtype) { return dtype == MIRL_DTYPE_BF16 || dtype == MIRL_DTYPE_F16; }

extern "C" int mirl_linear_ce_fwd(const void* hidden, int dtype, int64_t T, int64_t Hd, int64_t ldh,
                                  const void* weight, int64_t V, int64_t ldw, int64_t bsz,
                                  const int64_t* target, int64_t t_stride_b, int64_t t_stride_s,
                                  int64_t vocab_start, int64_t vocab_end, float* out,
                                  int64_t o_stride_b, int64_t o_stride_s, float* row_stats,
                                  float* workspace, void* stream) {
  clear_error();
  MIRL_REQUIRE(lce_dtype_ok(dtype), "hidden states and weight must be bf16 or fp16 (dtype code %d)",
               dtype);
  if (int e = check_common(hidden, T, Hd, ldh, weight, V, ldw, target, bsz)) return e;
  if (T == 0) return MIRL_OK;
  MIRL_REQUIRE(out && workspace, "null pointer argument");
  hipStream_t st = static_cast<hipStream_t>(stream);
  LceParams P{};
  P.h = static_cast<const uint16_t*>(hidden);
  P.w = static_cast<const uint16_t*>(weight);
  P.ldh = ldh;
  P.ldw = ldw;
  P.V = V;
  P.Hd = Hd;
  P.row0 = 0;
  P.nrows = T;
  P.bsz = bsz;
  P.target = target;
  P.tsb = t_stride_b;
  P.tss = t_stride_s;
  P.vs = vocab_start;
  P.ve = vocab_end;
  P.n_mt = ceil_div(T, kBM);
  P.n_nt = ceil_div(V, kBN);
  P.part = workspace;
  P.xt = workspace + T * P.n_nt * 2;
  const int64_t grid = ceil_div(P.n_mt * P.n_nt, kXcds) * kXcds;
  MIRL_REQUIRE(grid < (int64_t(1) << 31), "too many tiles");
  if (dtype == MIRL_DTYPE_BF16)
    hipLaunchKernelGGL((lce_tile_kernel<kFwd, BF16>), dim3((unsigned)grid), dim3(kThreads), 0, st, P);
  else
    hipLaunchKernelGGL((lce_tile_kernel<kFwd, F16>), dim3((unsigned)grid), dim3(kThreads), 0, st, P);
  hipLaunchKernelGGL(lce_merge_kernel, dim3((unsigned)ceil_div(T, 4)), dim3(256), 0, st, P.part,
                     P.xt, (int64_t)0, T, P.n_nt, bsz, target, t_stride_b, t_stride_s,
                     vocab_start, vocab_end, V, out, o_stride_b, o_stride_s, row_stats);
  return check_launch("mirl_linear_ce_fwd");
}

extern "C" int mirl_linear_ce_grad(const void* hidden, int dtype, int64_t T, int64_t Hd, int64_t ldh,
                                   const void* weight, int64_t V, int64_t ldw, int64_t bsz,
                                   const int64_t* target, int64_t t_stride_b,
                                   int64_t t_stride_s, int64_t vocab_start, int64_t vocab_end,
                                   const float* row_stats, const float* grad_out,
                                   int64_t g_stride_b, int64_t g_stride_s, int64_t row0,
                                   int64_t nrows, void* grad_logits, int64_t ldg,
                                   void* grad_logits_t, int64_t ldgt, const int64_t* row_count,
                                   void* stream) {
  clear_error();
  MIRL_REQUIRE(lce_dtype_ok(dtype), "hidden states and weight must be bf16 or fp16 (dtype code %d)",
               dtype);
  if (int e = check_common(hidden, T, Hd, ldh, weight, V, ldw, target, bsz)) return e;
  MIRL_REQUIRE(row0 >= 0 && nrows >= 0 && row0 + nrows <= T, "row range [%lld, %lld) outside [0, %lld)",
               (long long)row0, (long long)(row0 + nrows), (long long)T);
  if (nrows == 0) return MIRL_OK;
  MIRL_REQUIRE(row_stats && grad_out && grad_logits, "null pointer argument");
  MIRL_REQUIRE(ldg >= V, "gradient row stride %lld is smaller than V=%lld", (long long)ldg,
               (long long)V);
  // the transposed tiles cover whole 256-row tiles, written as 16-byte vectors
  MIRL_REQUIRE(grad_logits_t == nullptr ||
                   (ldgt >= ceil_div(nrows, kBM) * kBM && ldgt % 8 == 0 &&
                    (reinterpret_cast<uintptr_t>(grad_logits_t) & 15u) == 0),
               "transposed gradient: row stride %lld must cover %lld rows in whole 256-row tiles, "
               "be a multiple of 8 elements and start 16-byte aligned",
               (long long)ldgt, (long long)nrows);
  hipStream_t st = static_cast<hipStream_t>(stream);
  LceParams P{};
  P.h = static_cast<const uint16_t*>(hidden);
  P.w = static_cast<const uint16_t*>(weight);
  P.ldh = ldh;
  P.ldw = ldw;
  P.V = V;
  P.Hd = Hd;
  P.row0 = row0;
  P.nrows = nrows;
  P.bsz = bsz;
  P.target = target;
  P.tsb = t_stride_b;
  P.tss = t_stride_s;
  P.vs = vocab_start;
  P.ve = vocab_end;
  P.n_mt = ceil_div(nrows, kBM);
  P.n_nt = ceil_div(V, kBN);
  P.stats = row_stats;
  P.g = grad_out;
  P.gsb = g_stride_b;
  P.gss = g_stride_s;
  P.G = static_cast<uint16_t*>(grad_logits);
  P.ldg = ldg;
  P.Gt = static_cast<uint16_t*>(grad_logits_t);
  P.ldgt = ldgt;
  P.count = row_count;
  const int64_t grid = ceil_div(P.n_mt * P.n_nt, kXcds) * kXcds;
  MIRL_REQUIRE(grid < (int64_t(1) << 31), "too many tiles");
  if (dtype == MIRL_DTYPE_BF16)
    hipLaunchKernelGGL((lce_tile_kernel<kGrad, BF16>), dim3((unsigned)grid), dim3(kThreads), 0, st, P);
  else
    hipLaunchKernelGGL((lce_tile_kernel<kGrad, F16>), dim3((unsigned)grid), dim3(kThreads), 0, st, P);
  return check_launch("mirl_linear_ce_grad");
}

extern "C" int mirl_gemm_bf16_abt(const void* A, int64_t lda, const void* B, int64_t ldb, int64_t M,
                                  int64_t N, int64_t K, int64_t k_splits, float* C, int64_t ldc,
                                  int accumulate, void* Cb, int64_t ldcb, int cb_dtype,
                                  const int64_t* count, int64_t count_off, int count_axis,
                                  int64_t final_at, void* stream) {
  clear_error();
  MIRL_REQUIRE(Cb == nullptr || lce_dtype_ok(cb_dtype), "the 16-bit output must be bf16 or fp16 (dtype code %d)",
               cb_dtype);
  MIRL_REQUIRE(M >= 0 && N >= 0 && K > 0 && k_splits >= 1, "invalid shape M=%lld N=%lld K=%lld splits=%lld",
               (long long)M, (long long)N, (long long)K, (long long)k_splits);
  if (M == 0 || N == 0) return MIRL_OK;
  MIRL_REQUIRE(A && B && (C || Cb), "null pointer argument");
  const int64_t kstep = (int64_t)kStages * kSK;
  MIRL_REQUIRE(K % kstep == 0, "reduction length %lld must be a multiple of %lld", (long long)K,
               (long long)kstep);
  const int64_t kb = ceil_div(ceil_div(K, k_splits), kstep) * kstep;
  const int64_t n_ks = ceil_div(K, kb);
  MIRL_REQUIRE(n_ks == k_splits,
               "%lld splits of K=%lld in ranges of %lld leave %lld non-empty (choose a split count "
               "that divides into whole 128-element ranges)",
               (long long)k_splits, (long long)K, (long long)kb, (long long)n_ks);
  MIRL_REQUIRE(count_axis == MIRL_COUNT_ROWS || count_axis == MIRL_COUNT_K, "invalid count axis %d",
               count_axis);
  const bool both = C != nullptr && Cb != nullptr;
  MIRL_REQUIRE(!both || (count != nullptr && count_axis == MIRL_COUNT_K && n_ks == 1),
               "an fp32 and a bf16 output together take a reduction-length count and one split");
  MIRL_REQUIRE(Cb == nullptr || (n_ks == 1 && (!accumulate || both)),
               "a bf16 output takes one split and accumulates only over the fp32 output");
  MIRL_REQUIRE(!accumulate || n_ks == 1, "accumulation takes one split");
  MIRL_REQUIRE(lda % 8 == 0 && ldb % 8 == 0 && lda >= K && ldb >= K,
               "row strides (%lld, %lld) must be multiples of 8 elements and >= K", (long long)lda,
               (long long)ldb);
  MIRL_REQUIRE((reinterpret_cast<uintptr_t>(A) & 15u) == 0 && (reinterpret_cast<uintptr_t>(B) & 15u) == 0,
               "operands must be 16-byte aligned");
  // buffer ranges of one 256-row tile are 32-bit byte counts
  MIRL_REQUIRE(kBM * lda * 2 < (int64_t(1) << 31) && kBN * ldb * 2 < (int64_t(1) << 31),
               "row strides (%lld, %lld) too large", (long long)lda, (long long)ldb);
  MIRL_REQUIRE(M < (int64_t(1) << 31) && N < (int64_t(1) << 31), "sizes exceed 2^31-1");
  MIRL_REQUIRE(C == nullptr || ldc >= N, "output row stride %lld is smaller than N=%lld",
               (long long)ldc, (long long)N);
  MIRL_REQUIRE(Cb == nullptr || ldcb >= N, "output row stride %lld is smaller than N=%lld",
               (long long)ldcb, (long long)N);
  LceParams P{};
  P.h = static_cast<const uint16_t*>(A);
  P.w = static_cast<const uint16_t*>(B);
  P.ldh = lda;
  P.ldw = ldb;
  P.V = N;
  P.Hd = K;
  P.row0 = 0;
  P.nrows = M;
  P.n_mt = ceil_div(M, kBM);
  P.n_nt = ceil_div(N, kBN);
  P.n_ks = n_ks;
  P.kb_len = kb;
  P.C = C;
  P.Cb = static_cast<uint16_t*>(Cb);
  P.cb_f16 = cb_dtype == MIRL_DTYPE_F16;
  P.ldc = ldc;
  P.ldcb = ldcb;
  P.accumulate = accumulate;
  P.count = count;
  P.count_off = count_off;
  P.count_axis = count_axis;
  P.final_at = final_at;
  const int64_t grid = ceil_div(P.n_mt * P.n_nt * n_ks, kXcds) * kXcds;
  MIRL_REQUIRE(grid < (int64_t(1) << 31), "too many tiles");
  hipLaunchKernelGGL((lce_tile_kernel<kGemm, BF16>), dim3((unsigned)grid), dim3(kThreads), 0,
                     static_cast<hipStream_t>(stream), P);
  return check_launch("mirl_gemm_bf16_abt");
}

extern "C" int mirl_sum_splits_bf16(const float* part, int64_t k_splits, int64_t M, int64_t N,
                                    int64_t ld, void* out, int64_t ldo, int out_dtype,
                                    const int64_t* out_rows, int64_t out_nrows,
                                    const int64_t* count, int64_t count_off, void* stream) {
  clear_error();
  MIRL_REQUIRE(lce_dtype_ok(out_dtype) || out_dtype == MIRL_DTYPE_F32,
               "the output must be bf16, fp16 or fp32 (dtype code %d)", out_dtype);
  MIRL_REQUIRE(M >= 0 && N >= 0 && k_splits >= 1 && ld >= N && ldo >= N, "invalid shape");
  if (M == 0 || N == 0) return MIRL_OK;
  MIRL_REQUIRE(part && out, "null pointer argument");
  MIRL_REQUIRE(out_rows == nullptr || out_nrows >= 0, "invalid output row count");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uintptr_t out_align = out_dtype == MIRL_DTYPE_F32 ? 15u : 7u;  // 4 elements
  const bool vec4 = N % 4 == 0 && ld % 4 == 0 && ldo % 4 == 0 &&
                    (reinterpret_cast<uintptr_t>(part) & 15u) == 0 &&
                    (reinterpret_cast<uintptr_t>(out) & out_align) == 0;
  auto launch = [&](auto vec_c, auto eo) {
    constexpr int VEC = decltype(vec_c)::value;
    using EO = decltype(eo);
    hipLaunchKernelGGL((sum_splits_kernel<VEC, EO>), dim3((unsigned)ceil_div(M * N / VEC, 256)),
                       dim3(256), 0, st, part, k_splits, M, N, ld, out, ldo, out_rows, out_nrows,
                       count, count_off);
  };
  using V4 = std::integral_constant<int, 4>;
  using V1 = std::integral_constant<int, 1>;
  if (out_dtype == MIRL_DTYPE_BF16) {
    if (vec4) launch(V4{}, BF16{}); else launch(V1{}, BF16{});
  } else if (out_dtype == MIRL_DTYPE_F16) {
    if (vec4) launch(V4{}, F16{}); else launch(V1{}, F16{});
  } else {
    if (vec4) launch(V4{}, F32{}); else launch(V1{}, F32{});
  }
  return check_launch("mirl_sum_splits_bf16");
}

extern "C" int mirl_transpose_bf16(const void* src, int src_dtype, int64_t R, int64_t C,
                                   int64_t lds, void* dst, int64_t ldd, int64_t R_pad,
                                   const int64_t* count, void* stream) {
  clear_error();
  MIRL_REQUIRE(lce_dtype_ok(src_dtype), "the source must be bf16 or fp16 (dtype code %d)", src_dtype);
  MIRL_REQUIRE(R >= 0 && C >= 0 && R_pad >= R && lds >= C && ldd >= R_pad, "invalid shape");
  if (C == 0 || R_pad == 0) return MIRL_OK;
  MIRL_REQUIRE(src && dst, "null pointer argument");
  const int64_t n_rt = ceil_div(R_pad, 64), n_ct = ceil_div(C, 64);
  MIRL_REQUIRE(n_rt * n_ct < (int64_t(1) << 31), "too many tiles");
  auto launch = [&](auto es) {
    using ES = decltype(es);
    hipLaunchKernelGGL((transpose_bf16_kernel<ES>), dim3((unsigned)(n_rt * n_ct)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(src), R, C,
                       lds, static_cast<uint16_t*>(dst), ldd, R_pad, n_ct, count);
  };
  if (src_dtype == MIRL_DTYPE_BF16) launch(BF16{}); else launch(F16{});
  return check_launch("mirl_transpose_bf16");
}

extern "C" int mirl_gemm_f32_abt(const float* A, int64_t lda, const float* B, int64_t ldb, int64_t M,
                                 int64_t N, int64_t K, int64_t k_splits, float* C, int64_t ldc,
                                 int accumulate, const int64_t* count, int64_t count_off,
                                 int count_axis, void* stream) {
  clear_error();
  MIRL_REQUIRE(M >= 0 && N >= 0 && K > 0 && k_splits >= 1, "invalid shape M=%lld N=%lld K=%lld splits=%lld",
               (long long)M, (long long)N, (long long)K, (long long)k_splits);
  if (M == 0 || N == 0) return MIRL_OK;
  MIRL_REQUIRE(A && B && C, "null pointer argument");
  const int64_t kstep = (int64_t)kStages * (kRowBytes / 4);
  MIRL_REQUIRE(K % kstep == 0, "reduction length %lld must be a multiple of %lld", (long long)K,
               (long long)kstep);
  const int64_t kb = ceil_div(ceil_div(K, k_splits), kstep) * kstep;
  const int64_t n_ks = ceil_div(K, kb);
  MIRL_REQUIRE(n_ks == k_splits,
               "%lld splits of K=%lld in ranges of %lld leave %lld non-empty (choose a split count "
               "that divides into whole 64-element ranges)",
               (long long)k_splits, (long long)K, (long long)kb, (long long)n_ks);
  MIRL_REQUIRE(count_axis == MIRL_COUNT_ROWS || count_axis == MIRL_COUNT_K, "invalid count axis %d",
               count_axis);
  MIRL_REQUIRE(!accumulate || n_ks == 1, "accumulation takes one split");
  MIRL_REQUIRE(lda % 4 == 0 && ldb % 4 == 0 && lda >= K && ldb >= K,
               "row strides (%lld, %lld) must be multiples of 4 elements and >= K", (long long)lda,
               (long long)ldb);
  MIRL_REQUIRE((reinterpret_cast<uintptr_t>(A) & 15u) == 0 && (reinterpret_cast<uintptr_t>(B) & 15u) == 0,
               "operands must be 16-byte aligned");
  // buffer ranges of one 256-row tile are 32-bit byte counts
  MIRL_REQUIRE(kBM * lda * 4 < (int64_t(1) << 31) && kBN * ldb * 4 < (int64_t(1) << 31),
               "row strides (%lld, %lld) too large", (long long)lda, (long long)ldb);
  MIRL_REQUIRE(M < (int64_t(1) << 31) && N < (int64_t(1) << 31), "sizes exceed 2^31-1");
  MIRL_REQUIRE(ldc >= N, "output row stride %lld is smaller than N=%lld", (long long)ldc, (long long)N);
  LceParams P{};
  P.h = A;
  P.w = B;
  P.ldh = lda;
  P.ldw = ldb;
  P.V = N;
  P.Hd = K;
  P.row0 = 0;
  P.nrows = M;
  P.n_mt = ceil_div(M, kBM);
  P.n_nt = ceil_div(N, kBN);
  P.n_ks = n_ks;
  P.kb_len = kb;
  P.C = C;
  P.Cb = nullptr;
  P.ldc = ldc;
  P.accumulate = accumulate;
  P.count = count;
  P.count_off = count_off;
  P.count_axis = count_axis;
  P.final_at = 0;
  const int64_t grid = ceil_div(P.n_mt * P.n_nt * n_ks, kXcds) * kXcds;
  MIRL_REQUIRE(grid < (int64_t(1) << 31), "too many tiles");
  hipLaunchKernelGGL((lce_tile_kernel<kGemm, F32>), dim3((unsigned)grid), dim3(kThreads), 0,
                     static_cast<hipStream_t>(stream), P);
  return check_launch("mirl_gemm_f32_abt");
}

extern "C" int mirl_lce_active_rows(const float* grad_out, int64_t g_stride_b, int64_t g_stride_s,
                                    int64_t T, int64_t bsz, const int64_t* target,
                                    int64_t t_stride_b, int64_t t_stride_s, const float* row_stats,
                                    const void* hidden, int dtype, int64_t Hd, int64_t ldh,
                                    int64_t* perm, int64_t* count, int64_t* target_out,
                                    float* stats_out, float* grad_rows, void* hidden_out,
                                    void* stream) {
  clear_error();
  MIRL_REQUIRE(lce_dtype_ok(dtype) || dtype == MIRL_DTYPE_F32,
               "hidden states must be bf16, fp16 or fp32 (dtype code %d)", dtype);
  MIRL_REQUIRE(T >= 0 && Hd > 0 && bsz > 0 && ldh >= Hd, "invalid shape T=%lld H=%lld B=%lld", (long long)T,
               (long long)Hd, (long long)bsz);
  MIRL_REQUIRE(T % bsz == 0, "row count %lld is not a multiple of the batch size %lld", (long long)T,
               (long long)bsz);
  MIRL_REQUIRE(T < (int64_t(1) << 31) - 8 * kActThreads, "too many rows (%lld)", (long long)T);
  MIRL_REQUIRE(count != nullptr, "null pointer argument");
  MIRL_REQUIRE(T == 0 || (grad_out && target && row_stats && hidden && perm && target_out && stats_out &&
                          grad_rows && hidden_out),
               "null pointer argument");
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(lce_active_rows_kernel, dim3(1), dim3(kActThreads), 0, st, grad_out, g_stride_b,
                     g_stride_s, (uint32_t)T, (uint32_t)bsz, perm, grad_rows, count);
  if (T > 0) {
    const int64_t esz = dtype == MIRL_DTYPE_F32 ? 4 : 2;
    const uintptr_t both = reinterpret_cast<uintptr_t>(hidden) | reinterpret_cast<uintptr_t>(hidden_out);
    auto launch = [&](auto unit) {
      using UNIT = decltype(unit);
      constexpr int64_t n = sizeof(UNIT);
      hipLaunchKernelGGL(lce_gather_rows_kernel<UNIT>, dim3((unsigned)std::min(T, kGatherGrid)), dim3(256), 0,
                         st, perm, count, T, (uint32_t)bsz, target, t_stride_b, t_stride_s, row_stats,
                         static_cast<const UNIT*>(hidden), Hd * esz / n, ldh * esz / n, target_out,
                         stats_out, static_cast<UNIT*>(hidden_out));
    };
    if ((both & 15u) == 0 && Hd * esz % 16 == 0 && ldh * esz % 16 == 0)
      launch(vu4{});
    else if (esz == 4)
      launch(uint32_t{});
    else
      launch(uint16_t{});
  }
  return check_launch("mirl_lce_active_rows");
}

extern "C" int mirl_transpose_f32(const float* src, int64_t R, int64_t C, int64_t lds, float* dst,
                                  int64_t ldd, int64_t R_pad, const int64_t* count, int64_t count_off,
                                  void* stream) {
  clear_error();
  MIRL_REQUIRE(R >= 0 && C >= 0 && R_pad >= R && lds >= C && ldd >= R_pad, "invalid shape");
  if (C == 0 || R_pad == 0) return MIRL_OK;
  MIRL_REQUIRE(src && dst, "null pointer argument");
  const int64_t n_rt = ceil_div(R_pad, 64), n_ct = ceil_div(C, 64);
  MIRL_REQUIRE(n_rt * n_ct < (int64_t(1) << 31), "too many tiles");
  hipLaunchKernelGGL(transpose_f32_kernel, dim3((unsigned)(n_rt * n_ct)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), src, R, C, lds, dst, ldd, R_pad, n_ct, count,
                     count_off);
  return check_launch("mirl_transpose_f32");
}
