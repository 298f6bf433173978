// Convolution operands of the split-bf16 core (split_gemm.hpp).
#pragma once

#include "conv.hpp"
#include "split_gemm.hpp"

namespace ttrl {

// Input-gradient A of a residue class (LdConvDxA): row r is an input pixel, k =
// (jh, jw, o) with O a multiple of 32, so a step is 32 channels of one tap.
struct SaConvDx {
  LdConvDxA src;
  using Params = LdConvDxA::Params;
  struct Live {
    static constexpr bool EXACT = false, PERM = true, TABLE = false;
    Params q;
    __amdgpu_buffer_rsrc_t rs;
    struct Raw { f32x4 a, b; };
    struct Row { uint32_t off; int ohc, owc; };
    struct Kb { uint32_t off; int jh, jw; };
    __device__ __forceinline__ Row row(int r, int lg) const {
      const LdConvDxA::Live::Row x = LdConvDxA::Live{q, rs}.row(r);
      return Row{uint32_t(x.base) * 4u + uint32_t(lg) * 16u, x.ohc, x.owc};
    }
    __device__ __forceinline__ Kb kbase(int k0) const {
      const LdConvDxA::Live::Kp x = LdConvDxA::Live{q, rs}.kpos(__builtin_amdgcn_readfirstlane(k0));
      return Kb{uint32_t(x.off) * 4u, x.v ? x.jh : 1 << 28, x.jw};
    }
    __device__ __forceinline__ void issue(const Row& r, const Kb& k, Raw& f) const {
      const bool in = uint32_t(r.ohc - k.jh) < uint32_t(q.OH) && uint32_t(r.owc - k.jw) < uint32_t(q.OW);
      const uint32_t o = in ? r.off + k.off : kBad;
      f.a = ld_f4(rs, o);
      f.b = ld_f4(rs, o + 64u);
    }
    __device__ __forceinline__ void resolve(const Raw& f, f32x4& a, f32x4& b) const {
      a = f.a;
      b = f.b;
    }
  };
  __device__ __forceinline__ Live live(int grp) const {
    const LdConvDxA::Live l = src.live(grp);
    return Live{l.q, l.rs};
  }
};

// Input-gradient B (LdConvDxB): column n = c, k contiguous along o.
struct SbConvDx {
  LdConvDxB src;
  using Params = LdConvDxB::Params;
  struct Live {
    static constexpr bool COL = false;
    Params q;
    __amdgpu_buffer_rsrc_t rs;
    __device__ __forceinline__ uint32_t row(int n) const { return n < q.C ? uint32_t(n * q.O) * 4u : kBad; }
    __device__ __forceinline__ uint32_t kbase(int k0) const {
      return LdConvDxB::Live{q, rs}.kpos(__builtin_amdgcn_readfirstlane(k0)).off;
    }
    __device__ __forceinline__ float elem(int n, int k) const {
      return ld_f1(rs, row(n) + LdConvDxB::Live{q, rs}.kpos(k).off);
    }
  };
  __device__ __forceinline__ Live live(int grp) const {
    const LdConvDxB::Live l = src.live(grp);
    return Live{l.q, l.rs};
  }
};

// Input-gradient epilogue (EpConvDx); C a multiple of the columns a lane stores.
struct SeConvDx {
  static constexpr bool PARTIALS = false;
  EpConvDx src;
  struct Bound {
    EpConvDx::Bound b;
    __amdgpu_buffer_rsrc_t rc, rm;
    __device__ __forceinline__ uint32_t off(int r, int c) const {
      const int n = b.d_nhnw.div(r);
      const int rem = r - n * b.d_nhnw.d;
      const int i = b.d_nw.div(rem), j = rem - i * b.nw;
      const int ih = b.ih0 + b.S * i, iw = b.iw0 + b.S * j;
      return r < b.rows && c < b.C ? uint32_t(((n * b.H + ih) * b.W + iw) * b.C + c) * 4u : kBad;
    }
    __device__ __forceinline__ float alpha() const { return b.alpha; }
    __device__ __forceinline__ float beta() const { return b.beta; }
    __device__ __forceinline__ bool masked() const { return b.has_xm; }
    __device__ __forceinline__ bool accumulates() const { return b.beta != 0.f; }
  };
  __device__ __forceinline__ int rows(int grp) const { return src.rows(grp); }
  __device__ __forceinline__ Bound bind(int grp) const {
    const EpConvDx::Bound b = src.bound(grp);
    return Bound{b, b.rdx, b.rxm};
  }
};

// Weight-gradient A(r = patch index, k = pixel): a lane's 8 k are 8 pixels,
// whose byte offsets the workgroup tabulates; its row's offset in the patch
// is its own.  Vector patch layouts only (no padding); uint8 frames are exact
// in one bf16.
template <bool U8>
struct SaPatchT {
  ConvGeo g;
  const void* x;
  uint32_t xbytes;

  struct Params {
    ConvCore g;
    const void* x;
    uint32_t xbytes;
  };
  struct Live {
    static constexpr bool EXACT = U8, PERM = false, TABLE = true;
    Params q;
    __amdgpu_buffer_rsrc_t rs;
    struct Raw { f32x4 a, b; };
    using Row = uint32_t;
    __device__ __forceinline__ uint32_t row(int r, int) const { return tap_off(q.g, r); }
    __device__ __forceinline__ uint32_t offset(int m) const { return pixel_base(q.g, m); }
    __device__ __forceinline__ float one(uint32_t o) const {
      if constexpr (U8) return __uint_as_float(ld_u8(rs, o));
      else return ld_f1(rs, o);
    }
    __device__ __forceinline__ void issue(uint32_t row, const u32x4& o0, const u32x4& o1, Raw& f) const {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f.a[j] = one(row + o0[j]);
        f.b[j] = one(row + o1[j]);
      }
    }
    __device__ __forceinline__ void resolve(const Raw& f, f32x4& a, f32x4& b) const {
      a = f.a;
      b = f.b;
      if constexpr (U8)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          a[j] = float(__float_as_uint(f.a[j]));
          b[j] = float(__float_as_uint(f.b[j]));
        }
    }
  };
  __device__ __forceinline__ Live live(int) const {
    const Params q = pin_pod(Params{conv_core(g), x, xbytes});
    return Live{q, make_res(q.x, q.xbytes)};
  }
};

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// How the split core runs a weight gradient: K (the pixels) in `splits` parts
// of `kchunk`, as many as fill the device twice with 64-row tiles and as the
// room for partials and kMaxDwSplits (whoever sums them reads them all)
// allow.  splits 0: the FP32 core, for operands that do not fit (out channels
// in whole float4s) and for gradients too small to pay for more partials.  The
// lines, timed over first layers of 1 to 4 frames and float layers of 1 x 1 to
// 5 x 5 kernels at 8 to 2,048 images (FP32 / split us):
//   kSplitProducts, in products with the last tile's empty columns: first layer
//     of 4 frames at 19,200 pixels (157 M) 13.6 / 13.7, at 25,600 (210 M) 16.2 /
//     15.5; second layer at 5,184 (170 M) 13.7 / 14.9, at 7,776 (255 M) 17.9 /
//     15.8; third at 4,704 (173 M) 13.8 / 15.4, at 9,408 (347 M) 20.8 / 17.5.
//   kSplitArea, weight elements: a smaller weight has too few tiles for the
//     parts that kMaxDwSplits allows.  144 x 32 at 51,200 pixels 19.5 / 24.3, at
//     165,888 39.6 / 55.0; 192 x 32 at 41,472 21.4 / 22.0; 256 x 32 wins as above.
//     Bytes take half the products: 192 x 32 of three frames at 73,728 pixels
//     26.4 / 25.9, at 204,800 57.9 / 54.9, 64 x 32 at 294,912 39.8 / 74.7.
//   kSplitBank, where the partials stay in a bank and the FP32 core saves no
//     launch: the second layer's partials at 5,184 pixels (170 M) 9.6 / 8.6, the
//     third's at 4,704 (173 M) 9.6 / 8.7.  Of bytes (updates of a DQN, 24 to 100
//     images of 52 to 84): at 59 M 122 / 120, at 67 M 112.3 / 111, at 88 M 128 / 124,
//     at 105 M 133.2 / 132.1 (its launch 9.2 / 8.1, the optimizer step, which reads
//     twice the parts, 15.1 / 15.6); at 21 M 84 / 87, at 28 M 86 / 88.
// Twice the parts added one after another show where all products have one sign
// (error against float64 1.1e-7 to 1.3e-7, FP32 core 0.7e-7 to 1.5e-7); sums of
// either sign are the closer by 1.1 to 3 times.
constexpr int kMaxDwSplits = 64;
constexpr long kSplitProducts = 200'000'000, kSplitBank = 150'000'000, kSplitBankU8 = 40'000'000;
constexpr long kSplitArea = 8192, kSplitAreaU8 = 6144;
struct DwSplit {
  int fn = 0, splits = 0, kchunk = 0;
};
inline DwSplit dw_split(const ConvGeo& g, const float* dy, int ones, long room, bool bank) {
  DwSplit d;
  if (g.fp32_order || g.O % 4 || !aligned16(dy) || gemm_force_set()) return d;
  const int kp = g.C * g.KH * g.KW;
  d.fn = g.O > 32 ? 4 : 2;
  const long area = long(kp) * ceil_div(g.O, 16 * d.fn) * (16 * d.fn);
  if (area < (g.u8 ? kSplitAreaU8 : kSplitArea)) return d;
  if (area * g.M < (!bank ? kSplitProducts : g.u8 ? kSplitBankU8 : kSplitBank)) return d;
  const long tiles = long(ceil_div(kp, 64)) * ceil_div(g.O, 16 * d.fn);
  const long stages = ceil_div(g.M, kSplitKB);
  const long most = std::min({room / (long(kp + ones) * g.O), long(kMaxDwSplits), stages});
  const long want = std::min(most, std::max(2L, 512 / tiles));
  if (want < 2 || want * tiles < 128) return d;
  const long per = ceil_div(stages, want);
  d.splits = int(ceil_div(stages, per));
  d.kchunk = int(per) * kSplitKB;
  return d;
}

// Its launch: partials [splits][kp + ones][O] to `part`.
template <bool U8>
inline int run_dw_split(ttrl_ctx* ctx, const DwSplit& d, const ConvGeo& g, const void* x, const float* dy, int ones,
                        float* part, const char* name) {
  const SaPatchT<U8> la{g, x, input_bytes(g)};
  SbCol lb;  // B(k = m, n = o) = dZ[m][o]
  lb.p[0] = dy;
  lb.ld = lb.rows = g.O;
  lb.K = g.M;
  const int M = g.C * g.KH * g.KW;
  const SePartials ep{M};
  if (d.fn == 4) return launch_split<1, 4>(ctx, la, lb, ep, M, g.O, g.M, 1, name, ones, part, d.splits, d.kchunk);
  return launch_split<1, 2>(ctx, la, lb, ep, M, g.O, g.M, 1, name, ones, part, d.splits, d.kchunk);
}

// dw_split for a layer whose partials go to `bank`, or to the workspace past
// `reserved` floats at its end (bank null); never for the general patch path.
template <int MODE>
inline DwSplit conv_dw_splits(ttrl_ctx* ctx, const ConvGeo& g, const float* dy, const float* db, long reserved,
                              const float* bank, float** part = nullptr) {
  if constexpr (MODE == kPatchGeneral) return DwSplit{};
  long wsf = kGradBankFloats;
  float* to = const_cast<float*>(bank);
  if (!to) {
    to = ctx_workspace(ctx, &wsf);
    wsf -= reserved;
  }
  if (part) *part = to;
  return dw_split(g, dy, db ? 1 : 0, wsf, bank != nullptr);
}

// The weight gradient on the split core, if it takes it: its partials left in
// `bank` and described by *out (bank not null), or summed from the workspace.
template <int MODE>
inline bool conv_dw_split(ttrl_ctx* ctx, const ConvDwProblem<MODE>& p, const ConvGeo& g, const void* x, float x_scale,
                          const float* dy, float* dwt, float* db, long reserved, float* bank, ttrl_grad_source* out,
                          const char* name, int* rc) {
  if constexpr (MODE == kPatchGeneral) {
    return false;
  } else {
    float* part = nullptr;
    const DwSplit d = conv_dw_splits<MODE>(ctx, g, dy, db, reserved, bank, &part);
    if (!d.splits) return false;
    *rc = run_dw_split<MODE == kPatchU8Word>(ctx, d, g, x, dy, db ? 1 : 0, part, name);
    if (*rc != TTRL_OK) return true;
    if (bank) {
      GemmPlan plan{};
      plan.splits = d.splits;
      *out = conv_dw_source(g, x_scale, dwt, db, part, plan);
      return true;
    }
    FDiv dn;
    dn.set(p.q.N);
    const unsigned blocks = std::min(2048u, unsigned(long(p.q.M) * p.q.N / 256 + 1));
    hipLaunchKernelGGL((k_splitk_reduce<EpStore>), dim3(blocks, 1), dim3(256), 0, stream_of(ctx), part, p.ep, p.q.M,
                       p.q.N, d.splits, dn);
    *rc = check_launch(name);
    return true;
  }
}

// Whether the split core forms a layer's input gradient; `first` its problem of
// the first residue classes, which are the most and the largest.  The lines
// were timed over 1 x 1 to 5 x 5 kernels at 8 to 512 images.  Under kSplitTiles
// the FP32 core's smaller tiles fill the device better (FP32 / split us: the
// third Nature-CNN layer's at 122 tiles 13.3 / 15.6, at 162 19.3 / 15.7; 3 x 3 on
// 32 channels at 128 9.4 / 10.7, at 192 12.9 / 11.0; of 32 columns, 5 x 5 at 100
// 24.4 / 26.3, at 200 40.8 / 34.9).  K plays no part down to 32 (half a stage of
// zeros): 1 x 1 at 256 7.0 / 6.6, 2 x 2 in strides of 2 at 576 12.0 / 9.6.
constexpr long kSplitTiles = 150;
inline bool dx_on_split(const ConvGeo& g, const ConvDxProblem& first) {
  return !g.fp32_order && g.O % 32 == 0 && g.C % 4 == 0 && !gemm_force_set() && aligned16(first.la.dy) &&
         aligned16(first.lb.wt) && aligned16(first.ep.dx) && aligned16(first.ep.xmask) &&
         split_tiles(first.q.M, first.q.N, first.q.groups) >= kSplitTiles;
}

// The input gradient, kMaxGroups residue classes a launch, all on one core.
inline int conv_dx(ttrl_ctx* ctx, const ConvGeo& g, const float* dy, const float* wt, float* dx, const float* xmask,
                   float x_scale, float beta, long reserved, const char* name) {
  bool split = false;
  int rc = TTRL_OK;
  for (int c0 = 0; c0 < g.S * g.S && rc == TTRL_OK; c0 += kMaxGroups) {
    const ConvDxProblem p = conv_dx_problem(g, c0, dy, wt, dx, xmask, x_scale, beta);
    if (c0 == 0) split = dx_on_split(g, p);
    if (split)
      rc = run_split(ctx, SaConvDx{p.la}, SbConvDx{p.lb}, SeConvDx{p.ep}, p.q.M, p.q.N, p.q.K, p.q.groups, name);
    else
      rc = run_gemm<kConvDxCfgs>(ctx, p.la, p.lb, p.ep, p.q.M, p.q.N, p.q.K, p.q.groups, name, reserved);
  }
  return rc;
}

}  // namespace ttrl
