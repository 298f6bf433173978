// FP32 products on the bf16 matrix cores of gfx950.
//
// A float is exactly the sum of three bf16 numbers: the float rounded to the
// nearest bf16, what is left rounded likewise, and the rest (8 significant
// bits each, either sign; Henry, Tang and Heinecke, "Leveraging the bfloat16
// Artificial Intelligence Datatype For Higher-Precision Computations", ARITH
// 2019).  A product of two floats is then nine bf16 products, of which the six
// largest are kept, each exact in FP32 and added in FP32 by the matrix core.
// The parts are at most 2^-8 and 2^-17 of the operand's power of two, so what
// is left out is at most 2^-24 + 2^-34 of the product, of either sign, and
// 16x16x32 bf16 MFMA runs six of them in 3/8 of the time 16x16x4 FP32 MFMA
// takes for the product.  (Parts cut off instead of rounded leave out up to
// 2^-21, always towards zero: a sum of positive terms came out 0.69 * 2^-24
// low, rounded parts leave its mean error at 0.005 * 2^-24.)  Bytes (uint8
// frames) are exact in one bf16, so they take three.
//
// What it gives (both gradients of a Nature-CNN layer, batch 256; FP32 core
// before): second layer 62.2 -> 45.4 us, third 50.5 -> 39.4; batch 1024 and 512
// 196.5 -> 118.4 and 88.1 -> 55.1.  The error against float64 falls, since the
// main sum is rounded once per 32 k: weight gradients at batch 1024 6.9e-7 ->
// 2.2e-7, input gradients 2.7e-7 -> 8.5e-8, at K = 32 (2 x 2 kernels, stride 2)
// 1.0e-7 -> 3.9e-8.  What bounds it: a stage's chain of loads, splits (5.5 VALU
// instructions per float) and LDS round trips; the matrix core is busy 10 to 12 %
// of the time at batch 256, 23 % at 1024.
//
// One workgroup owns BM x BN of the output, NW wavefronts along M, each
// WM x FN fragments of 16 x 16.
//   A: every wavefront owns its rows, so nothing is shared: each lane loads
//      the 8 consecutive k of its fragment row (two 16-byte loads) straight
//      into registers two 32-deep steps ahead and splits them there.
//   B: shared by the wavefronts: staged KB deep through LDS, split once per
//      workgroup, in three planes of 16-byte units (8 k of one column), the
//      unit of column n at slot (n % FN) * 16 + n / FN, so that a lane's FN
//      fragments are FN consecutive columns (vector stores), two buffers, one
//      barrier a stage.
//
// Infinities, NaN and values whose sums overflow do not survive the split
// (inf - inf), and operands under 2^-110 lose their lowest bits (bf16 ends at
// 2^-133).  A wavefront that finds a non-finite sum, or no sum of kSplitTiny in
// its tile, forms the tile again with FP32 MFMA, whose results it then stores,
// so such inputs give what the FP32 core gives; what small operands lose beside
// larger ones is under 2^-134 of the other operand.  A tile of exact zeros stays
// (masked gradients are often zero throughout), so sums whose every operand
// lies under 2^-134, below float32's normal range, may vanish.
#pragma once

#include "tile_gemm.hpp"

namespace ttrl {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t hi_pair(float a, float b) {  // upper halves of (a, b), a in the low half
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
// (a, b) to the nearest bf16 pair, left as a's and b's rest (exact).
__device__ __forceinline__ uint32_t take_nearest(float& a, float& b) {
  uint32_t p = __builtin_bit_cast(uint32_t, bf16x2{__bf16(a), __bf16(b)});  // v_cvt_pk_bf16_f32
  asm("" : "+v"(p));  // else the lower half is converted again on its own
  a -= __uint_as_float(p << 16);
  b -= __uint_as_float(p & 0xffff0000u);
  return p;
}

// The three planes of a pair of floats.
__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = take_nearest(a, b);
  m = take_nearest(a, b);
  l = hi_pair(a, b);  // at most 8 significant bits are left
}

struct Planes {
  u32x4 h, m, l;
};
template <bool EXACT>
__device__ __forceinline__ void split8(const f32x4& a, const f32x4& b, Planes& p) {
  if constexpr (EXACT) {
    p.h = u32x4{hi_pair(a.x, a.y), hi_pair(a.z, a.w), hi_pair(b.x, b.y), hi_pair(b.z, b.w)};
  } else {
    uint32_t h[4], m[4], l[4];
    split2(a.x, a.y, h[0], m[0], l[0]);
    split2(a.z, a.w, h[1], m[1], l[1]);
    split2(b.x, b.y, h[2], m[2], l[2]);
    split2(b.z, b.w, h[3], m[3], l[3]);
    p.h = u32x4{h[0], h[1], h[2], h[3]};
    p.m = u32x4{m[0], m[1], m[2], m[3]};
    p.l = u32x4{l[0], l[1], l[2], l[3]};
  }
}

__device__ __forceinline__ f32x4 mfma_bf16(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}

// ---------------------------------------------------------- A operands ---
//
// live(g) as for the FP32 core's loaders.  A step is 32 k.  row(m, lg): the
// address part of one output row for lane group lg; issue: starts a lane's
// loads; resolve: its 8 values.  Addresses along k are kbase(k0), of the step
// from k0 (wave-uniform; K a multiple of 32), or with TABLE offset(k), of one k
// (any K); both take any k and past K make every address out of range, so that
// such elements read zero.  With PERM lane group lg holds k = 4 lg .. 4 lg + 3
// and 16 + 4 lg .. of the step, so each load takes 64 contiguous bytes of a row
// from its four lanes; without, k = 8 lg .. 8 lg + 7.  B is stored to match.

// ---------------------------------------------------------- B operands ---
//
// Vector loads only, no element paths: a branch in the loop that only some
// lanes take makes the wavefront wait for its loads where the branch joins,
// one memory round trip per fetch.  COL (n contiguous): at(n, k) is the byte
// offset of the four elements from (n, k), kbytes() the bytes from k to k + 1;
// offsets only grow, so past K they run out of the operand's range and read
// zeros.  Otherwise (k contiguous) row(n) + kbase(k0) addresses the 32 k of
// the step from k0, as for A.

// v(n, k) = p[g][k*ld + n]; four n a load: rows a multiple of 4, 16-byte rows.
struct SbCol {
  const float* p[kMaxGroups] = {};
  long ld = 0;
  int rows = 0, K = 0;
  __host__ __device__ long bytes() const { return K > 0 && rows > 0 ? ((long(K) - 1) * ld + rows) * 4 : 0; }
  struct Params {
    const float* p;
    uint32_t bytes;
    int ld, rows, K;
  };
  struct Live {
    static constexpr bool COL = true;
    Params q;
    __amdgpu_buffer_rsrc_t rs;
    __device__ __forceinline__ uint32_t at(int n, int k) const {
      return n < q.rows ? uint32_t(k * q.ld + n) * 4u : kBad;
    }
    __device__ __forceinline__ uint32_t kbytes() const { return uint32_t(q.ld) * 4u; }
    __device__ __forceinline__ float elem(int n, int k) const {
      return ld_f1(rs, n < q.rows && k < q.K ? uint32_t(k * q.ld + n) * 4u : kBad);
    }
  };
  __device__ __forceinline__ Live live(int g) const {
    const Params q = pin_pod(Params{p[g], uint32_t(bytes()), int(ld), rows, K});
    return Live{q, make_res(q.p, q.bytes)};
  }
};

// ----------------------------------------------------------- epilogues ---
//
// A lane stores FN consecutive columns of a row at once; n is a multiple of
// FN and so are the output's columns and row pitch.  v = alpha*acc (* [mask > 0])
// (+ beta*old), the mask and the old value read only where there is one.
template <int N>
using FVec = float __attribute__((ext_vector_type(N)));

template <int N>
__device__ __forceinline__ FVec<N> ld_vec(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  if constexpr (N == 4) return ld_f4(r, off);
  else return __builtin_bit_cast(FVec<2>, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
__device__ __forceinline__ void st_vec(__amdgpu_buffer_rsrc_t r, uint32_t off, const FVec<4>& v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, 0);
}
__device__ __forceinline__ void st_vec(__amdgpu_buffer_rsrc_t r, uint32_t off, const FVec<2>& v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, 0, 0);
}
// Row r of a fragment row's FN fragments.
template <int FN>
__device__ __forceinline__ FVec<FN> row_of(const f32x4 (&a)[FN], int r) {
  FVec<FN> v;
#pragma unroll
  for (int j = 0; j < FN; ++j) v[j] = a[j][r];
  return v;
}

// No epilogue: partials of K, which their reader sums.
struct SePartials {
  static constexpr bool PARTIALS = true;
  int M = 0;
  __device__ __forceinline__ int rows(int) const { return M; }
};

// ------------------------------------------------------------ the core ---

template <int BN, int KB>
struct SplitLds {
  static constexpr int KG = KB / 8;
  static constexpr int KGS = BN + 2;             // units per k-group: the two spare units spread the banks
  static constexpr int PLANE = KG * KGS;         // units
  static constexpr int BUF = 3 * PLANE;
  static constexpr int UNITS = 2 * BUF;
};

// One stage of B in flight and its way into LDS.  PERM: the k order of A's
// lane groups (above).
template <int BN, int FN, int KB, int NT, bool PERM, class VB, bool COL = VB::COL>
struct BStage;

// The 8-byte half of the unit that holds k quad kq of column n.
template <int BN, int FN, int KB, bool PERM>
__device__ __forceinline__ u32x2* b_slot(u32x4* lds, int n, int kq) {
  using L = SplitLds<BN, KB>;
  const int kg = PERM ? (kq >> 3) * 4 + (kq & 3) : kq >> 1, half = PERM ? (kq >> 2) & 1 : kq & 1;
  return reinterpret_cast<u32x2*>(lds + kg * L::KGS + (n % FN) * 16 + n / FN) + half;
}

// n contiguous (four columns a load): a unit is four columns x four k.
template <int BN, int FN, int KB, int NT, bool PERM, class VB>
struct BStage<BN, FN, KB, NT, PERM, VB, true> {
  static constexpr int CH = BN / 4, UNITS = CH * (KB / 4), PER = (UNITS + NT - 1) / NT;
  static constexpr bool WHOLE = UNITS % NT == 0;
  uint32_t off[PER];
  f32x4 f[PER][4];
  f32x4 sum[PER];  // of each column over the k this thread stages, in order
  __device__ __forceinline__ void init(const VB& vb, int n0, int k0, int tid) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int i = tid + u * NT;
      off[u] = vb.at(n0 + (i % CH) * 4, k0 + (i / CH) * 4);
      sum[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  __device__ __forceinline__ void add(int piece) {
    const int u = piece / 4, j = piece % 4;
    sum[u][j] += (f[u][0][j] + f[u][1][j]) + (f[u][2][j] + f[u][3][j]);
  }
  // The workgroup's column sums: row kq of red[KB / 4][BN].
  __device__ __forceinline__ void put_sums(float* red, int tid) const {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int i = tid + u * NT;
      if (WHOLE || i < UNITS) *reinterpret_cast<f32x4*>(red + (i / CH) * BN + (i % CH) * 4) = sum[u];
    }
  }
  // Loads the next stage.
  __device__ __forceinline__ void issue(const VB& vb, int, int tid) {
    const uint32_t kb = vb.kbytes();
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      if (WHOLE || tid + u * NT < UNITS)
#pragma unroll
        for (int r = 0; r < 4; ++r) f[u][r] = ld_f4(vb.rs, off[u] + uint32_t(r) * kb);
      off[u] += KB * kb;
    }
  }
  // Piece j of PIECES (one of a thread's columns) into LDS.
  static constexpr int PIECES = PER * 4;
  __device__ __forceinline__ void write(u32x4* lds, int piece, int tid) {
    using L = SplitLds<BN, KB>;
    const int u = piece / 4, j = piece % 4;
    const int i = tid + u * NT, c = i % CH, kq = i / CH;
    if (!WHOLE && i >= UNITS) return;
    uint32_t h0, m0, l0, h1, m1, l1;
    split2(f[u][0][j], f[u][1][j], h0, m0, l0);
    split2(f[u][2][j], f[u][3][j], h1, m1, l1);
    u32x2* d = b_slot<BN, FN, KB, PERM>(lds, 4 * c + j, kq);
    d[0] = u32x2{h0, h1};
    d[2 * L::PLANE] = u32x2{m0, m1};
    d[4 * L::PLANE] = u32x2{l0, l1};
  }
};

// k contiguous: a unit is one column x four k.
template <int BN, int FN, int KB, int NT, bool PERM, class VB>
struct BStage<BN, FN, KB, NT, PERM, VB, false> {
  static constexpr int CH = KB / 4, PER = BN * CH / NT, PIECES = PER;
  static_assert(KB == 64 && NT % CH == 0 && BN * CH % NT == 0, "two steps a stage, whole units per thread");
  uint32_t row[PER];
  f32x4 f[PER];
  __device__ __forceinline__ void init(const VB& vb, int n0, int, int tid) {
#pragma unroll
    for (int u = 0; u < PER; ++u) row[u] = vb.row(n0 + (tid + u * NT) / CH) + uint32_t(tid % CH & 7) * 16u;
  }
  // Loads the stage from k0.
  __device__ __forceinline__ void issue(const VB& vb, int k0, int tid) {
    const uint32_t s0 = vb.kbase(k0), s1 = vb.kbase(k0 + 32);
    const uint32_t kb = tid % CH < CH / 2 ? s0 : s1;
#pragma unroll
    for (int u = 0; u < PER; ++u) f[u] = ld_f4(vb.rs, row[u] + kb);
  }
  __device__ __forceinline__ void write(u32x4* lds, int u, int tid) {
    using L = SplitLds<BN, KB>;
    uint32_t h0, m0, l0, h1, m1, l1;
    split2(f[u].x, f[u].y, h0, m0, l0);
    split2(f[u].z, f[u].w, h1, m1, l1);
    u32x2* d = b_slot<BN, FN, KB, PERM>(lds, (tid + u * NT) / CH, tid % CH);
    d[0] = u32x2{h0, h1};
    d[2 * L::PLANE] = u32x2{m0, m1};
    d[4 * L::PLANE] = u32x2{l0, l1};
  }
};

constexpr int kSplitKB = 64;
// With operands up to 2^16 on the other side and 2^12 terms, 2^-134 of them is
// under 2^-24 of this.
constexpr float kSplitTiny = 0x1p-80f;

template <int WM, int FN, int NW, class LA, class LB, class EP>
__global__ __launch_bounds__(64 * NW) void k_split(LA la, LB lb, EP ep, float* ws, int M, int N, int K, int kchunk,
                                                   int splits, int ones) {
  constexpr int KB = kSplitKB, NT = 64 * NW, BM = NW * WM * 16, BN = FN * 16, KS = KB / 32;
  using L = SplitLds<BN, KB>;
  using VA = typename LA::Live;
  using VB = typename LB::Live;
  __shared__ __attribute__((aligned(16))) u32x4 lds[L::UNITS];
  __shared__ __attribute__((aligned(16))) uint32_t table[VA::TABLE ? 2 : 1][VA::TABLE ? KB : 4];
  warm_kernargs<int(sizeof(LA) + sizeof(LB) + sizeof(EP) + sizeof(float*) + 6 * sizeof(int))>();
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = int(blockIdx.z) / splits, split = int(blockIdx.z) - g * splits;
  const int m0 = int(blockIdx.x) * BM, n0 = int(blockIdx.y) * BN;
  if (m0 >= ep.rows(g)) return;  // uniform per block: ragged residue classes
  const int kbeg = split * kchunk, kend = min(K, kbeg + kchunk);
  const int lr = lane & 15, lg = lane >> 4;
  const int mw = m0 + wave * (WM * 16);

  const VA va = la.live(g);
  const VB vb = lb.live(g);
  // A: loads one stage ahead, the split one step ahead of its products.
  BStage<BN, FN, KB, NT, VA::PERM, VB> bs;
  typename VA::Row ra[WM];
  typename VA::Raw fa[KS][WM];
  Planes pa[KS][WM];
  bs.init(vb, n0, kbeg, tid);
  bs.issue(vb, kbeg, tid);
  // Where A's 8 k of a lane are 8 places in memory, the workgroup finds a
  // stage's KB addresses together, two stages ahead.
  if constexpr (VA::TABLE) {
    if (tid < 2 * KB) table[tid / KB][tid % KB] = va.offset(kbeg + tid);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < WM; ++i) ra[i] = va.row(mw + i * 16 + lr, lg);
  auto issue_a = [&](int s, int k0) {
    if constexpr (VA::TABLE) {
      const uint32_t* t = table[((k0 - kbeg) / KB) & 1] + s * 32 + lg * 8;
#pragma unroll
      for (int i = 0; i < WM; ++i) va.issue(ra[i], *reinterpret_cast<const u32x4*>(t), *reinterpret_cast<const u32x4*>(t + 4), fa[s][i]);
    } else {
      const auto kb = va.kbase(k0 + s * 32);
#pragma unroll
      for (int i = 0; i < WM; ++i) va.issue(ra[i], kb, fa[s][i]);
    }
  };
  auto split_a = [&](int s, int i) {
    f32x4 x, y;
    va.resolve(fa[s][i], x, y);
    split8<VA::EXACT>(x, y, pa[s][i]);
  };
#pragma unroll
  for (int s = 0; s < KS; ++s) issue_a(s, kbeg);
  f32x4 acc[WM][FN], low[WM][FN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = low[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int q = 0; q < bs.PIECES; ++q) {
    bs.write(lds, q, tid);
    if constexpr (VB::COL)
      if (ones) bs.add(q);
  }
  bs.issue(vb, kbeg + KB, tid);
#pragma unroll
  for (int i = 0; i < WM; ++i) split_a(0, i);
  __syncthreads();
  // One stage is one basic block (loads and splits past the end read zeros,
  // or in a split of K the next part's operands, and are not used) in NB
  // pieces, each the products of two columns of fragments over one step with
  // a share of the next splits in front.  B's next stage is written in the
  // first half, so that the loads after it have the other half and more.
  constexpr int NB = KS * FN / 2;
  int buf = 0;
  for (int k0 = kbeg; k0 < kend; k0 += KB) {
    const u32x4* T = lds + buf * L::BUF + lg * L::KGS + lr;
    buf ^= 1;
    u32x4* W = lds + buf * L::BUF;
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int s = q / (FN / 2), jp = q % (FN / 2) * 2;
      u32x4 bh[2], bm[2], bl[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const u32x4* t = T + s * 4 * L::KGS + (jp + c) * 16;
        bh[c] = t[0];
        bm[c] = t[L::PLANE];
        bl[c] = t[2 * L::PLANE];
      }
      if (jp == 0) issue_a(s, k0 + KB);
#pragma unroll
      for (int i = 0; i < WM; ++i)
        if (i * (FN / 2) / WM == jp / 2) split_a((s + 1) % KS, i);
#pragma unroll
      for (int w = 0; w < bs.PIECES; ++w)
        if (w * (NB / 2) / bs.PIECES == q) {
          bs.write(W, w, tid);
          if constexpr (VB::COL)
            if (ones && k0 + KB < kend) bs.add(w);
        }
      if (q + 1 == NB / 2) bs.issue(vb, k0 + 2 * KB, tid);
      const Planes(&a)[WM] = pa[s];
      // Product by product, so that consecutive MFMAs are independent.  The
      // products of the lower parts have sums of their own (2^-8 of the
      // whole), so the main sum is rounded once per 32 k.
      auto product = [&](f32x4 (&d)[WM][FN], auto part, const u32x4 (&pb)[2]) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int i = 0; i < WM; ++i) d[i][jp + c] = mfma_bf16(a[i].*part, pb[c], d[i][jp + c]);
      };
      if constexpr (!VA::EXACT) product(low, &Planes::l, bh);
      product(acc, &Planes::h, bh);
      if constexpr (!VA::EXACT) product(low, &Planes::m, bm);
      product(low, &Planes::h, bl);
      if constexpr (!VA::EXACT) product(low, &Planes::m, bh);
      product(low, &Planes::h, bm);
    }
    if constexpr (VA::TABLE)  // into the half that the stage before this one read
      if (tid < KB) table[((k0 - kbeg) / KB) & 1][tid] = va.offset(k0 + 2 * KB + tid);
    __syncthreads();
  }

  bool finite = true;
  float top = 0.f;
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        acc[i][j][r] += low[i][j][r];
        finite = finite && __builtin_isfinite(acc[i][j][r]);
        top = fmaxf(top, fabsf(acc[i][j][r]));
      }
  if (!__all(finite) || (__any(top > 0.f) && !__any(top >= kSplitTiny))) {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int k0 = kbeg; k0 < kend; k0 += 32) {
      f32x4 x[WM][2];
#pragma unroll
      for (int i = 0; i < WM; ++i) {
        typename VA::Raw f;
        if constexpr (VA::TABLE) {
          u32x4 o0, o1;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            o0[j] = va.offset(k0 + lg * 8 + j);
            o1[j] = va.offset(k0 + lg * 8 + 4 + j);
          }
          va.issue(ra[i], o0, o1, f);
        } else {
          va.issue(ra[i], va.kbase(k0), f);
        }
        va.resolve(f, x[i][0], x[i][1]);
      }
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const float b = vb.elem(n0 + FN * lr + j, k0 + (VA::PERM ? (s >> 2) * 16 + lg * 4 + (s & 3) : lg * 8 + s));
#pragma unroll
          for (int i = 0; i < WM; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i][s >> 2][s & 3], b, acc[i][j], 0, 0, 0);
        }
    }
  }

  const int n = n0 + FN * lr;
  if constexpr (EP::PARTIALS) {
    const int prows = M + ones;  // a partial's rows: the column sums below the product
    float* const part = ws + (long(g) * splits + split) * prows * N;
    if (ones && blockIdx.x == 0) {
      float* red = reinterpret_cast<float*>(lds);  // the loop ended with a barrier
      bs.put_sums(red, tid);
      __syncthreads();
      if (tid < BN && n0 + tid < N) {
        float t = 0.f;
#pragma unroll
        for (int q = 0; q < KB / 4; ++q) t += red[q * BN + tid];
        part[long(M) * N + n0 + tid] = t;
      }
    }
    const __amdgpu_buffer_rsrc_t rw = make_res(part, uint32_t(M) * uint32_t(N) * 4u);
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = mw + i * 16 + 4 * lg + r;
        st_vec(rw, m < M && n < N ? (uint32_t(m) * uint32_t(N) + uint32_t(n)) * 4u : kBad, row_of<FN>(acc[i], r));
      }
  } else {
    const auto eb = ep.bind(g);
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      uint32_t off[4];
      FVec<FN> keep[4], old[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) off[r] = eb.off(mw + i * 16 + 4 * lg + r, n);
      if (eb.masked())
#pragma unroll
        for (int r = 0; r < 4; ++r) keep[r] = ld_vec<FN>(eb.rm, off[r]);
      if (eb.accumulates())
#pragma unroll
        for (int r = 0; r < 4; ++r) old[r] = ld_vec<FN>(eb.rc, off[r]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        FVec<FN> v = row_of<FN>(acc[i], r);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          v[j] *= eb.alpha();
          if (eb.masked() && !(keep[r][j] > 0.f)) v[j] = 0.f;
          if (eb.accumulates()) v[j] += eb.beta() * old[r][j];
        }
        st_vec(eb.rc, off[r], v);
      }
    }
  }
}

// ---------------------------------------------------------------- host ---

// The split core's tile for a GEMM: rows of a workgroup (64 or 128; wm = 1, 2
// fragments a wavefront) by 16 fn columns.  Of the two heights the one with the
// shorter last wave of workgroups, 64 rows costing 0.55 of 128 (third Nature-CNN
// layer's input gradient at batch 512, 648 tiles of 64 or 324 of 128: 27.9 / 30.1
// us; second layer's, 3200 or 1600: 37.6 / 36.2).
struct SplitTile {
  int wm = 0, fn = 0;
};
SplitTile split_tile(long M, long N, long groups);
long split_tiles(long M, long N, long groups);  // its 64 x 64 tiles, those of 32 columns counted half

template <int WM, int FN, class LA, class LB, class EP>
inline int launch_split(ttrl_ctx* ctx, const LA& la, const LB& lb, const EP& ep, int M, int N, int K, int groups,
                        const char* name, int ones, float* ws, int splits, int kchunk) {
  constexpr int NW = 4;
  const dim3 grid(ceil_div(M, NW * WM * 16), ceil_div(N, FN * 16), unsigned(groups * splits));
  hipLaunchKernelGGL((k_split<WM, FN, NW, LA, LB, EP>), grid, dim3(64 * NW), 0, stream_of(ctx), la, lb, ep, ws, M, N, K,
                     kchunk, splits, ones);
  return check_launch(name);
}

template <class LA, class LB, class EP>
inline int run_split(ttrl_ctx* ctx, const LA& la, const LB& lb, const EP& ep, int M, int N, int K, int groups,
                     const char* name) {
  const SplitTile t = split_tile(M, N, groups);
  const int kchunk = int(ceil_div(K, kSplitKB)) * kSplitKB;
  auto go = [&](auto wm, auto fn) {
    return launch_split<decltype(wm)::value, decltype(fn)::value>(ctx, la, lb, ep, M, N, K, groups, name, 0, nullptr, 1,
                                                                  kchunk);
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I4 = std::integral_constant<int, 4>;
  if (t.fn == 4) return t.wm == 2 ? go(I2{}, I4{}) : go(I1{}, I4{});
  return t.wm == 2 ? go(I2{}, I2{}) : go(I1{}, I2{});
}

}  // namespace ttrl
