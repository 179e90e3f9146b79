// gemm_mfma.hip — the MFMA-tiled complex GEMM for products of more than 64
// rows (the prompt pass and training): multiply_complex (utils/matrix.rs:16-65)
// with the epilogues of epilogue.hpp and the fused greedy id.
//
// This file is compiled on its own with -mllvm -amdgpu-mfma-vgpr-form=1
// (rustcrates_amd/build.py).  By default the compiler kept the accumulators
// in AGPRs for the MFMAs but carried them across the K loop in VGPRs, so every
// K step copied all of them back (v_accvgpr_write) and waited for the tile
// loads before the first MFMA.  In the VGPR form the loop has no copies.  The
// flag is kept to this file: the skinny decode products measured slower with it.
#include "epilogue.hpp"
#include "train.hpp"

namespace mitok {

// ===========================================================================
// C[M][N] = A[M][K] B[K][N], bound by the FP64 matrix cores.
//
// Block tile 64x64, 8 waves of 32x16, K step 8.  Per 16x16x4 step a wave
// issues, per output tile, the v_mfma_f64_16x16x4_f64 of
//     Cr += Ar*Br;  Ci += Ar*Bi;  Cr -= Ai*Bi;  Ci += Ai*Br
// (signs as MFMA modifiers).  An operand known to be real (the rows a Norm
// leaves, a softmax gradient, the gradient of a Norm's input) takes only the
// two products its real part is in, and EPI_RE only Cr's two: half the
// matrix work of a complex product, which is what these launches spend their
// time on.  The products left out are with zeros; only 0 * (infinity or NaN)
// would show, so each thread keeps the largest exponent of what it stages of
// the other operand and the result becomes NaN where that is not finite: every
// result is what the four products give.
//
// Why this tile: a wave step is 64 cycles per MFMA, so the loop is bound by how
// well loads and barriers hide behind it.  With 80 registers a wave (the real
// QKV form and seven of backward's spill 1 to 3 more) and 32 KB of LDS a block,
// three blocks (six waves per SIMD) share a CU and one's barrier is covered by
// another's MFMAs; global loads go out two K steps
// ahead into registers, fragments one 4-k step ahead.  Measured on MI355X
// (TFLOP/s at 8, real A 4 flops per complex multiply-add), against 64x64 with
// 4 waves of 32x32, K step 16, one step ahead:
//     16384 x 3072 x 768   62.4 -> 72.0, real A 31 -> 66.8
//     4096 x 1536 x 512    53.6 -> 68.8, real A 30 -> 63.0
//     2048 x 512 x 2048    50.7 -> 64.1, real A 25 -> 55.8
// (torch's complex matmul reaches 74.6 at 4096 cubed).  64x128 and 128x128
// tiles and 4 waves of 32x32 were within 2% at the largest shape and slower
// wherever the grid is short.
//
// Lane layout of v_mfma_f64_16x16x4_f64 (wave64): A[i][k] at lane i+16k,
// B[k][j] at lane j+16k, D[i][j] at lane j+16*(i%4), element i/4 (unlike the
// f32 16x16x4 form, consecutive output rows sit in consecutive lane groups).
//
// Operands (GemmOpnd, train.hpp): a row-major complex or double array as it
// is or transposed, conjugated or not, real or not.  Backward's products read
// their transposes in place; each materialised one cost a pass over memory
// and a launch.
// ===========================================================================
constexpr int GNT = 512;  // threads
constexpr int GMT = 2;    // 16-row tiles of a wave
__device__ const double2 gemm_zero2 = {0.0, 0.0};  // what a load outside the operand reads

// One operand's 64 x 8 tile in LDS.  ALONG_K: the stored array is contiguous
// along K (A as it is, B transposed): element (i, k) at row i, its k XORed so
// that the 16 rows of a fragment fall in different banks.  Else contiguous
// along the tile's rows or columns (A transposed, B as it is): [k][64], doubles
// with odd k shifted half a bank row.
template <int F, bool ALONG_K>
struct GemmTile {
  static constexpr bool real = (F & (OP_RE | OP_F64)) != 0;
  static constexpr bool f64 = (F & OP_F64) != 0;
  typedef typename std::conditional<real, double, double2>::type T;    // in LDS
  typedef typename std::conditional<f64, double, double2>::type TG;   // in memory
  static constexpr int BYTES = GBM * GBK * (int)sizeof(T);
  static __device__ __forceinline__ int slot(int i, int k) {
    if constexpr (ALONG_K) return i * GBK + (k ^ (real ? 2 * ((i >> 2) & 3) : ((i >> 1) & 7)));
    else return k * GBM + (real ? i ^ ((k & 1) << 4) : i);
  }
  const TG* p;   // this thread's element of the next K step
  long step;     // elements from one K step to the next
  int left;      // K elements left for it (0: outside the operand)
  int at;        // its slot in LDS
  __device__ __forceinline__ void init(const void* base, long ld, int i0, int n, int kbeg, int kend, int tid) {
    const int i = ALONG_K ? tid / GBK : tid % GBM, k = ALONG_K ? tid % GBK : tid / GBM;
    const long ii = min(i0 + i, n - 1), kk = kbeg + k;
    p = (const TG*)base + (ALONG_K ? ii * ld + kk : kk * ld + ii);
    step = ALONG_K ? GBK : (long)GBK * ld;
    left = i0 + i < n ? kend - kbeg - k : 0;
    at = slot(i, k);
  }
  __device__ __forceinline__ T next() {
    const TG v = ld_glb(left > 0 ? p : (const TG*)&gemm_zero2);
    p += step;
    left -= GBK;
    if constexpr (real && !f64) return v.x;
    else return v;
  }
};
__device__ __forceinline__ double re_of(double v) { return v; }
__device__ __forceinline__ double re_of(double2 v) { return v.x; }
__device__ __forceinline__ double im_of(double) { return 0.0; }
__device__ __forceinline__ double im_of(double2 v) { return v.y; }
template <bool NEG>  // c + a b, or c - a b
__device__ __forceinline__ v4d mfma64(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, NEG ? 1 : 0);
}

// Tile t of an mt x nt grid: (row, column).  Blocks go to the 8 XCDs in turn
// and each XCD has its own L2.  Where one side is short its tiles run fastest
// within the blocks of one XCD, so that a column (or row) of tiles, with its
// slice of the larger operand, belongs to one XCD and is read once: 1024 x
// 32000 x 512, whose 262 MB of weights row order streams 16 times, 2000 ->
// 1932 us, real A 1191 -> 1116; 4096 x 512 x 2048 498 -> 488.  A tall grid of
// more columns than an XCD's blocks cover twice goes row by row (16384 x 3072
// x 768, real A: 2415 us, 2523 by rows of an XCD).
constexpr int TALL_MAX_COLS = 16;
__device__ __forceinline__ int2 tile_at(int t, int mt, int nt) {
  const bool wide = nt > mt;
  if (!wide && nt > TALL_MAX_COLS) return make_int2(t / nt, t % nt);
  const int major = wide ? nt : mt, minor = wide ? mt : nt, even = major / 8 * 8;
  int a, b;
  if (t < even * minor) {
    const int j = t >> 3;
    a = j / minor * 8 + (t & 7), b = j % minor;
  } else {
    const int r = t - even * minor;
    a = even + r / minor, b = r % minor;
  }
  return wide ? make_int2(b, a) : make_int2(a, b);
}

// MODE: the epilogue mode, fixed at compile time so each launch carries only
// its own epilogue.  AF, BF: how the operands are read.  Of the tiles in
// tile_at's order the first `whole` are one block each, every later
// one is `splits` blocks of kchunk of K whose last to arrive sums the
// partials in split order.
template <int MODE, int AF, int BF>
__global__ __launch_bounds__(GNT, 6) void k_zgemm_mfma(const void* __restrict__ A, long lda, const void* __restrict__ Bm,
                                                       long ldb, int M, int N, int K, int whole, int splits,
                                                       int kchunk, Epi ep_in, Argmax am, double2* __restrict__ ws,
                                                       uint32_t* __restrict__ cnt, MfmaBatch bt) {
  using TA = GemmTile<AF, !(AF & OP_T)>;
  using TB = GemmTile<BF, (BF & OP_T) != 0>;
  constexpr bool RE = MODE == EPI_RE;  // only the real part is used
  static_assert(!(TA::real && TB::real), "one operand is complex");
  Epi ep = ep_in;
  ep.mode = MODE;
  if (bt.n > 1) {
    const long z = blockIdx.y, z0 = z / bt.inner, z1 = z - z0 * bt.inner, c = z0 * bt.c0 + z1 * bt.c1;
    A = (const typename TA::TG*)A + z0 * bt.a0 + z1 * bt.a1;
    Bm = (const typename TB::TG*)Bm + z0 * bt.b0 + z1 * bt.b1;
    if (RE) ep.out_re += c;
    else ep.out += c;
  }
  constexpr int STAGE = RE ? GBM * 65 * (int)sizeof(double) : 0;  // Re values of the tile for the fused argmax
  constexpr int TILES = 2 * (TA::BYTES + TB::BYTES);
  __shared__ __align__(16) char lds[TILES > STAGE ? TILES : STAGE];
  const auto As = [&](int st) { return (typename TA::T*)(lds + st * TA::BYTES); };
  const auto Bs = [&](int st) { return (typename TB::T*)(lds + 2 * TA::BYTES + st * TB::BYTES); };
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i = lane & 15, kq = lane >> 4;
  const int nt = (N + GBN - 1) / GBN, tiles = nt * ((M + GBM - 1) / GBM);
  int tile = blockIdx.x, split = 0, kbeg = 0, kend = K;
  if (tile >= whole) {
    const int r = tile - whole, rest = tiles - whole;
    split = r / rest;
    tile = whole + (r - split * rest);
    kbeg = split * kchunk;
    kend = min(K, kbeg + kchunk);
  }
  const int2 pos = tile_at(tile, tiles / nt, nt);
  const int m0 = pos.x * GBM, n0 = pos.y * GBN;
  const int wm = (wave >> 2) * 32, wn = (wave & 3) * 16;

  TA ta;
  TB tb;
  ta.init(A, lda, m0, M, kbeg, kend, tid);
  tb.init(Bm, ldb, n0, N, kbeg, kend, tid);
  typename TA::T ra[2], fa[2][GMT];
  typename TB::T rb[2], fb[2];
  // where one operand is real: the largest high words (sign off) of the other's real and imaginary parts
  int top_re = 0, top_im = 0;
  auto gload = [&](int s) {
    ra[s] = ta.next();
    rb[s] = tb.next();
  };
  auto sstore = [&](int st, int s) {
    As(st)[ta.at] = ra[s];
    Bs(st)[tb.at] = rb[s];
    if constexpr (TA::real || TB::real) {
      const double re = TA::real ? re_of(rb[s]) : re_of(ra[s]), im = TA::real ? im_of(rb[s]) : im_of(ra[s]);
      top_re = max(top_re, __double2hiint(re) & 0x7fffffff);
      top_im = max(top_im, __double2hiint(im) & 0x7fffffff);
    }
  };
  auto frag = [&](int st, int kk, int f) {
#pragma unroll
    for (int t = 0; t < GMT; ++t) fa[f][t] = As(st)[TA::slot(wm + 16 * t + i, kk + kq)];
    fb[f] = Bs(st)[TB::slot(wn + i, kk + kq)];
  };
  v4d cr[GMT], ci[GMT];
#pragma unroll
  for (int t = 0; t < GMT; ++t) cr[t] = ci[t] = v4d{0.0, 0.0, 0.0, 0.0};
  // a conjugated operand's imaginary part enters with the other sign
  constexpr bool NA = (AF & OP_CJ) != 0, NB = (BF & OP_CJ) != 0;
  auto mma = [&](int f) {
#pragma unroll
    for (int t = 0; t < GMT; ++t) {
      const double ar = re_of(fa[f][t]), br = re_of(fb[f]);
      cr[t] = mfma64<false>(ar, br, cr[t]);
      if constexpr (!RE && !TB::real) ci[t] = mfma64<NB>(ar, im_of(fb[f]), ci[t]);
      if constexpr (!RE && TB::real) ci[t] = mfma64<NA>(im_of(fa[f][t]), br, ci[t]);
    }
    // every tile's first products before any tile's last ones: an
    // accumulator's next MFMA is never adjacent to its previous one
    if constexpr (!TA::real && !TB::real) {
#pragma unroll
      for (int t = 0; t < GMT; ++t) {
        const double ai = im_of(fa[f][t]);
        cr[t] = mfma64<NA == NB>(ai, im_of(fb[f]), cr[t]);
        if constexpr (!RE) ci[t] = mfma64<NA>(ai, re_of(fb[f]), ci[t]);
      }
    }
  };

  const int nk = kend > kbeg ? (kend - kbeg + GBK - 1) / GBK : 0;
  gload(0);  // steps past the last load zeros
  gload(1);
  sstore(0, 0);
  gload(0);
  __syncthreads();
  frag(0, 0, 0);
  auto step = [&](int st) {  // K step in LDS half st; the next one is in register stage st ^ 1
    frag(st, 4, 1);
    mma(0);
    mma(1);
    sstore(st ^ 1, st ^ 1);
    gload(st ^ 1);
    // with half the MFMAs per step the loads must not sink below the barrier
    // (4096 x 512 x 2048, real A: 57.4 -> 59.6 TFLOP/s; a complex product
    // measured 1% slower with the order fixed)
    if constexpr (TA::real || TB::real) __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    frag(st ^ 1, 0, 0);
  };
  for (int it = 0; it < nk; it += 2) {
    step(0);
    if (it + 1 >= nk) break;
    step(1);
  }

  if constexpr (TA::real || TB::real) {
    // column (real A) or row (real B) of the tile -> whether its sums meet 0 * (infinity or NaN):
    // the real sum with the imaginary parts, the imaginary sum with the real ones
    __shared__ int bad[2][GBM];
    if (tid < GBM) bad[0][tid] = bad[1][tid] = 0;
    __syncthreads();
    const int mine = (TA::real ? (BF & OP_T) != 0 : !(AF & OP_T)) ? tid / GBK : tid % GBM;
    if (top_im >= 0x7ff00000) bad[0][mine] = 1;
    if (top_re >= 0x7ff00000) bad[1][mine] = 1;
    __syncthreads();
    if constexpr (TA::real)
      if (bt.zero_row && m0 == 0 && tid < GBN && n0 + tid < N) {
        // no MFMA forms this row, so the 0 * (infinity or NaN) they would meet shows here too
        if (bad[0][tid] || bad[1][tid]) bt.zero_row[n0 + tid] = make_double2(NAN, NAN);
      }
#pragma unroll
    for (int t = 0; t < GMT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int at = TA::real ? wn + i : wm + 16 * t + 4 * e + kq;
        if (bad[0][at]) cr[t][e] = NAN;
        if (bad[1][at]) ci[t][e] = NAN;
      }
  }

  if (blockIdx.x >= (unsigned)whole && splits > 1) {
    // partials of (tile, split), one run of 512 elements per accumulator element
    const long base = (long)(tile - whole) * splits;
    double2* mine = ws + (base + split) * (GBM * GBN) + tid;
#pragma unroll
    for (int t = 0; t < GMT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) st_dev(mine + (t * 4 + e) * GNT, make_double2(cr[t][e], ci[t][e]));
    if (!arrive_last(&cnt[tile - whole], (uint32_t)splits)) return;
    for (int p = 0; p < splits; ++p) {
      const double2* part = ws + (base + p) * (GBM * GBN) + tid;
#pragma unroll
      for (int t = 0; t < GMT; ++t) {
        double2 v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = ld_dev(part + (t * 4 + e) * GNT);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          cr[t][e] = p ? cr[t][e] + v[e].x : v[e].x;
          ci[t][e] = p ? ci[t][e] + v[e].y : v[e].y;
        }
      }
    }
  }
  const bool argmax = RE && am.part_v != nullptr;
  double* stage = (double*)lds;  // [64][65], the operand tiles are consumed
#pragma unroll
  for (int t = 0; t < GMT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int ml = wm + 16 * t + 4 * e + kq, nl = wn + i;
      const int m = m0 + ml, n = n0 + nl;
      if (m < M && n < N) {
        double2 v = make_double2(cr[t][e], ci[t][e]);
        if (MODE == EPI_STORE && bt.scale != 1.0) v = cscale(v, bt.scale);
        const double re = apply_epi(ep, M, N, m, n, v);
        if constexpr (RE)
          if (argmax) stage[ml * 65 + nl] = re;
      }
    }
  if constexpr (RE) {
    if (!argmax) return;
    __syncthreads();
    // per-row (max, last index) over the tile's columns: wave w takes rows w, w + 8, ...
    for (int ml = wave; ml < GBM; ml += GNT / 64) {
      const int m = m0 + ml, n = n0 + lane;
      if (m >= M) break;
      double bv = -INFINITY;
      int bi = -1;
      if (n < N) {
        const double v = stage[ml * 65 + lane];
        if (isnan(v)) atomicOr(am.err, (uint32_t)EB_ARGMAX_NAN);
        else bv = v, bi = n;
      }
      wave_argmax(bv, bi);
      if (lane == 0) {
        am.part_v[(long)m * nt + pos.y] = bv;
        am.part_i[(long)m * nt + pos.y] = bi;
      }
    }
  }
}

template <int MODE, int AF, int BF>
static int launch(hipStream_t st, const MfmaPlan& p, const GemmOpnd& A, const GemmOpnd& B, int M, int N, int K,
                  const Epi& ep, const Argmax& am, double2* ws, uint32_t* cnt, const MfmaBatch& bt) {
  MITOK_LAUNCH((k_zgemm_mfma<MODE, AF, BF>), dim3((unsigned)p.blocks(), (unsigned)bt.n), dim3(GNT), 0, st, A.p, A.ld,
               B.p, B.ld, M, N, K, p.whole, p.P, p.kchunk, ep, am, ws, cnt, bt);
  return OK;
}

int launch_zgemm_mfma(hipStream_t st, const MfmaPlan& p, const GemmOpnd& A, const GemmOpnd& B, int M, int N, int K,
                      const Epi& ep, const Argmax& am, double2* ws, uint32_t* cnt, const MfmaBatch& bt) {
  if (bt.n < 1 || bt.n > 65535 || (bt.n > 1 && p.P > 1)) return ERR_ARG;  // a batch has no split workspace
  const auto key = [](int mode, int a, int b) { return mode << 8 | a << 4 | b; };
#define MITOK_CASE(MODE, AF, BF) \
  case MODE << 8 | (AF) << 4 | (BF): return launch<MODE, AF, BF>(st, p, A, B, M, N, K, ep, am, ws, cnt, bt);
  switch (key(ep.mode, A.flags, B.flags)) {
    // the forward pass: rows times weights
    MITOK_CASE(EPI_STORE, 0, 0)
    MITOK_CASE(EPI_STORE, OP_RE, 0)
    MITOK_CASE(EPI_GELU, 0, 0)
    MITOK_CASE(EPI_GELU, OP_RE, 0)
    MITOK_CASE(EPI_RE, 0, 0)
    MITOK_CASE(EPI_RE, OP_RE, 0)
    MITOK_CASE(EPI_QKV, 0, 0)
    MITOK_CASE(EPI_QKV, OP_RE, 0)
    // weight gradients conj(X)^T G
    MITOK_CASE(EPI_STORE, OP_H, 0)
    MITOK_CASE(EPI_STORE, OP_H | OP_RE, 0)
    MITOK_CASE(EPI_STORE, OP_H, OP_RE)
    MITOK_CASE(EPI_STORE, OP_H, OP_F64)
    // input gradients G conj(W)^T
    MITOK_CASE(EPI_STORE, 0, OP_H)
    MITOK_CASE(EPI_STORE, OP_RE, OP_H)
    MITOK_CASE(EPI_STORE, OP_F64, OP_H)
    // attention: Re(Q K^T), Re(G conj(V)^T), dA conj(K), dA^T conj(Q), A^T G
    MITOK_CASE(EPI_RE, 0, OP_T)
    MITOK_CASE(EPI_RE, 0, OP_H)
    MITOK_CASE(EPI_STORE, OP_F64, OP_CJ)
    MITOK_CASE(EPI_STORE, OP_F64 | OP_T, OP_CJ)
    MITOK_CASE(EPI_STORE, OP_F64 | OP_T, 0)
    default: return ERR_ARG;
  }
#undef MITOK_CASE
}

}  // namespace mitok
