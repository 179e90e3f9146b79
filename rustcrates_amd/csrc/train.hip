// train.hip — backward's kernels on gfx950 around its tiled products
// (gemm_mfma.hip): SoftmaxLayer::backward (softmax_output_layer.rs:67-145),
// LinearLayer::backward's sums (linear_layer.rs:77-128) and update_parameters
// (:130-175) with the reference's AdamW (utils/adam_w.rs:9-103), and the
// elementwise and row kernels of the other layers' reverse walk.
//
//   G  = softmax gradient (p - [c == target]) / (B * non-PAD targets of b) of
//        the rows that predict a target (the host maps rows to targets); the
//        other rows' is zero.  The head's products run on the target rows
//        alone, packed, with one zero row standing for all the others
//   dW = conj(X)^T G and dX = G conj(W)^T, transposes read in place
//   db = the column sums of G
//   update: the first update descends by lr * clip(g) / B where finite; later
//        ones run AdamW on the unclipped grouped gradient (AdamW clips each
//        element to norm 1 itself), moments kept per parameter.
#include "train.hpp"

namespace mitok {

// Packed row i of the softmax gradient, real: (p - [c == target]) / norm of
// output row rows[i], or the zero row (rows[i] < 0).  One block per row.
__global__ __launch_bounds__(256) void k_softmax_grad(const double* __restrict__ P, int V, const int* __restrict__ rows,
                                                      const int* __restrict__ tgt, const double* __restrict__ norm,
                                                      int S, double* __restrict__ G) {
  const long i = blockIdx.x;
  const int r = rows[i], t = r < 0 ? -1 : tgt[r];
  const double nz = r < 0 ? 1.0 : norm[r / S];
  const double* p = P + (long)max(r, 0) * V;
  double* g = G + i * V;
  for (int c = threadIdx.x; c < V; c += 256) g[c] = t < 0 ? 0.0 : (c == t ? p[c] - 1.0 : p[c]) / nz;  // softmax_output_layer.rs:128-135
}

// Packed rows of X beside them: row r goes to packed[r].  The rows without a
// target share packed row `zero` (zeros before the launch): their gradient is
// zero, so all they could give a sum is the NaN of 0 * (infinity or NaN).
__global__ __launch_bounds__(256) void k_pack_rows(const double2* __restrict__ X, int d, const int* __restrict__ packed,
                                                   int zero, double2* __restrict__ out) {
  const long r = blockIdx.x;
  const int i = packed[r];
  for (int c = threadIdx.x; c < d; c += 256) {
    const double2 v = X[r * d + c];
    if (i != zero) {
      out[(long)i * d + c] = v;
    } else {
      if (!isfinite(v.x)) out[(long)i * d + c].x = NAN;
      if (!isfinite(v.y)) out[(long)i * d + c].y = NAN;
    }
  }
}

// out[r] = in[packed[r]]: the input gradient of every row from the packed ones
__global__ __launch_bounds__(256) void k_unpack_rows(const double2* __restrict__ in, int d,
                                                     const int* __restrict__ packed, double2* __restrict__ out) {
  const long r = blockIdx.x;
  const double2* src = in + (long)packed[r] * d;
  for (int c = threadIdx.x; c < d; c += 256) out[r * d + c] = src[c];
}

// db[c] = sum over sequences b of (sum over the rows s of b of G[s][c])
// (linear_layer.rs:101-105, group_gradient_batch_bias).  Bound by the loads in
// flight: a block takes 64 columns of one sequence, each wave a quarter of its
// rows, eight loads at a time, the quarters added in row order (8 x 128 rows of
// 2048: 18 -> 5.5 us against one thread per (sequence, column)).  Then one thread
// per column adds the sequences in order, times `mult`.  starts: sequence b's
// rows are [starts[b], starts[b + 1]), or null for S rows each.
__device__ __forceinline__ double zero_of(double) { return 0.0; }
__device__ __forceinline__ double2 zero_of(double2) { return make_double2(0.0, 0.0); }
__device__ __forceinline__ double addt(double a, double b) { return a + b; }
__device__ __forceinline__ double2 addt(double2 a, double2 b) { return cadd(a, b); }
template <class T>
__global__ __launch_bounds__(256) void k_seq_colsum(const T* __restrict__ G, const int* __restrict__ starts, int S,
                                                    int V, T* __restrict__ part) {
  __shared__ T quarter[3][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, cols = (V + 63) / 64;
  const int b = blockIdx.x / cols, c = (blockIdx.x - b * cols) * 64 + lane;
  const int r0 = starts ? starts[b] : b * S, n = (starts ? starts[b + 1] : r0 + S) - r0;
  const int ra = (int)((long)n * wave / 4), rb = (int)((long)n * (wave + 1) / 4);
  T s = zero_of(T());
  if (c < V) {
    const T* g = G + (long)(r0 + ra) * V + c;
    int r = ra;
    for (; r + 8 <= rb; r += 8) {
      T u[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) u[q] = g[(long)q * V];
#pragma unroll
      for (int q = 0; q < 8; ++q) s = addt(s, u[q]);
      g += 8l * V;
    }
    for (; r < rb; ++r, g += V) s = addt(s, g[0]);
  }
  if (wave) quarter[wave - 1][lane] = s;
  __syncthreads();
  if (wave == 0 && c < V) part[(long)b * V + c] = addt(addt(addt(s, quarter[0][lane]), quarter[1][lane]), quarter[2][lane]);
}
__device__ __forceinline__ double2 as_complex(double v) { return make_double2(v, 0.0); }
__device__ __forceinline__ double2 as_complex(double2 v) { return v; }
template <class T>
__global__ __launch_bounds__(256) void k_seq_sum(const T* __restrict__ part, int B, int V, double mult,
                                                 double2* __restrict__ out) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= V) return;
  T acc = zero_of(T());
  for (int b = 0; b < B; ++b) acc = addt(acc, part[(long)b * V + c]);
  out[c] = mult == 1.0 ? as_complex(acc) : cscale(as_complex(acc), mult);
}

// f64::powi as compiler-rt's __powidf2 (square and multiply over the bits)
__device__ __forceinline__ double powi_f64(double a, int e) {
  const bool recip = e < 0;
  double r = 1.0;
  for (;;) {
    if (e & 1) r *= a;
    e /= 2;
    if (e == 0) break;
    a *= a;
  }
  return recip ? 1.0 / r : r;
}

// One parameter: the first update's clipped descent (linear_layer.rs:159-174,
// clip_gradient_1d at utils/matrix.rs:709-717), or AdamW (adam_w.rs:9-103;
// `weight`: v_hat's norm at least EPSILON, which the bias arm omits).  This
// file is built with -ffp-contract=off: every multiply and add rounds on its
// own, as the Rust expressions do.
__device__ __forceinline__ double2 update1(double2 w, double2 g, double2* m, double2* v, const TrainStep& ts,
                                           bool weight) {
  if (ts.first) {
    // the descent stores zero moments for the AdamW that follows it
    // (linear_layer.rs:141-145,176-180): after reset_previous_gradient too
    *m = make_double2(0.0, 0.0);
    *v = make_double2(0.0, 0.0);
    const double n = hypot(g.x, g.y);
    if (n > 1.0) g = cscale(g, 1.0 / n);
    if (!(isfinite(g.x) && isfinite(g.y))) return w;
    return csub(w, cscale(cunscale(g, ts.batch), ts.lr));
  }
  const double B1 = 0.9, B2 = 0.999, EPS = 1e-8, WD = 0.01, MAX_NORM = 1.0;
  const int t = ts.time_step > 0 ? ts.time_step : 1;
  const double gn = hypot(g.x, g.y);
  if (gn > MAX_NORM) g = cscale(g, MAX_NORM / gn);
  const double2 mm = cadd(cscale(*m, B1), cscale(g, 1.0 - B1));
  const double2 vv = cadd(cscale(*v, B2), cmul(cscale(g, 1.0 - B2), make_double2(g.x, -g.y)));
  *m = mm;
  *v = vv;
  const double2 mh = cunscale(mm, 1.0 - powi_f64(B1, t));
  const double2 vh = cunscale(vv, 1.0 - powi_f64(B2, t));
  double vn = hypot(vh.x, vh.y);
  if (weight) vn = fmax(vn, EPS);
  const double alr = ts.lr / (sqrt(vn) + EPS);
  return csub(cscale(w, 1.0 - ts.lr * WD), cmul(make_double2(alr, 0.0), mh));
}

__global__ __launch_bounds__(256) void k_linear_update(double2* __restrict__ W, const double2* __restrict__ dW,
                                                       double2* __restrict__ mW, double2* __restrict__ vW, long n,
                                                       double2* __restrict__ b, const double2* __restrict__ db,
                                                       double2* __restrict__ mb, double2* __restrict__ vb, int V,
                                                       TrainStep ts) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) W[i] = update1(W[i], dW[i], &mW[i], &vW[i], ts, true);
  if (i < V) b[i] = update1(b[i], db[i], &mb[i], &vb[i], ts, false);
}

// gelu_derivative_complex (utils/derivative.rs:48-84): powi(3) = z (z z),
// powi(2) = t t; saturated beyond |f(z)| = 20; the result kept to norms in
// [1e-12, 1e6]
__device__ __forceinline__ double2 gelu_deriv(double2 z) {
  const double s2p = sqrt(2.0 / M_PI);
  const double2 one = make_double2(1.0, 0.0);
  const double2 x3 = cmul(z, cmul(z, z));
  const double2 fx = cscale(cadd(z, cmul(make_double2(0.044715, 0.0), x3)), s2p);
  const bool sat = hypot(fx.x, fx.y) > 20.0;
  const double2 th = sat ? one : ctanh_nc(fx);
  const double2 sech2 = sat ? make_double2(0.0, 0.0) : csub(one, cmul(th, th));
  const double2 fp = cscale(cadd(one, cmul(make_double2(0.134145, 0.0), cmul(z, z))), s2p);
  const double2 d = cadd(cmul(make_double2(0.5, 0.0), cadd(one, th)),
                         cmul(cmul(cmul(make_double2(0.5, 0.0), z), sech2), fp));
  const double n = hypot(d.x, d.y);
  if (n > 1e6) return cmul(cunscale(d, n), make_double2(1e6, 0.0));
  if (n < 1e-12) return make_double2(1e-12, 0.0);
  return d;
}

// Dense (GELU) backward's elementwise step (layer.rs:181-192): the gradient
// of the activated output, its padded rows zeroed (apply_padding_mask_batch),
// times conj(GELU'(Z)) of the pre-activation Z
__global__ __launch_bounds__(256) void k_gelu_backward(const double2* __restrict__ dH, const double2* __restrict__ Z,
                                                       const uint32_t* __restrict__ mask, long rows, int F,
                                                       double2* __restrict__ G) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= rows * F) return;
  const long r = i / F;
  double2 g = make_double2(0.0, 0.0);
  if (!mask || mask[r] != 0) {
    const double2 dz = gelu_deriv(Z[i]);
    g = cmul(dH[i], make_double2(dz.x, -dz.y));
  }
  G[i] = g;
}

void gelu_backward(hipStream_t st, const double2* dH, const double2* Z, const uint32_t* mask, long rows, int F,
                   double2* G) {
  const long n = rows * F;
  if (n > 0) MITOK_LAUNCH(k_gelu_backward, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dH, Z, mask, rows, F, G);
}

void softmax_grad(hipStream_t st, const double* P, int n, int V, const int* rows, const int* tgt, const double* norm,
                  int S, double* G) {
  if (n > 0) MITOK_LAUNCH(k_softmax_grad, dim3(n), dim3(256), 0, st, P, V, rows, tgt, norm, S, G);
}

void pack_rows(hipStream_t st, const double2* X, long rows, int d, const int* packed, int zero, double2* out) {
  fill_const(st, out + (long)zero * d, d, make_double2(0.0, 0.0));
  if (rows > 0) MITOK_LAUNCH(k_pack_rows, dim3((unsigned)rows), dim3(256), 0, st, X, d, packed, zero, out);
}

void unpack_rows(hipStream_t st, const double2* in, long rows, int d, const int* packed, double2* out) {
  if (rows > 0) MITOK_LAUNCH(k_unpack_rows, dim3((unsigned)rows), dim3(256), 0, st, in, d, packed, out);
}

// cross_entropy_loss_batch (transformer_network.rs:662-711) on the softmax
// output P [B][S][V].  Block b: its targets' terms -ln(p + 1e-15), p at row
// S - tl - 1 + t, are formed in parallel into LDS (PAD targets, id 1, marked
// skipped), then one thread sums them in target order and divides by their
// count (cross_entropy_loss, :674-711; no target is left out by its
// `seq_ind >= end_ind` break, since the rows end at S - 2).  part[b] holds it.
__global__ __launch_bounds__(256) void k_ce_seq(const double* __restrict__ P, int S, int V,
                                                const uint32_t* __restrict__ tgt, const uint32_t* __restrict__ tlen,
                                                int T, double* __restrict__ part) {
  extern __shared__ double lp[];  // [T]
  const int b = blockIdx.x, tl = (int)tlen[b];
  const int start = S - tl - 1;
  for (int t = threadIdx.x; t < tl; t += 256) {
    const uint32_t tc = tgt[(long)b * T + t];
    lp[t] = tc == 1u ? NAN : -log(P[((long)b * S + start + t) * V + tc] + 1e-15);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double loss = 0.0, count = 0.0;
    for (int t = 0; t < tl; ++t)
      if (tgt[(long)b * T + t] != 1u) {
        loss += lp[t];
        count += 1.0;
      }
    part[b] = loss / count;
  }
}

// the batch: sum of the sequences' losses in order, divided by B, as the
// complex (sum / B, 0 / B) the reference returns
__global__ void k_ce_batch(const double* __restrict__ part, int B, double* __restrict__ out) {
  if (threadIdx.x != 0) return;
  double re = 0.0;
  for (int b = 0; b < B; ++b) re += part[b];
  out[0] = re / (double)B;
  out[1] = 0.0 / (double)B;
}

void cross_entropy(hipStream_t st, const double* P, int B, int S, int V, const uint32_t* tgt, const uint32_t* tlen,
                   int T, double* part, double* out) {
  if (B <= 0) return;
  MITOK_LAUNCH(k_ce_seq, dim3(B), dim3(256), (size_t)T * sizeof(double), st, P, S, V, tgt, tlen, T, part);
  MITOK_LAUNCH(k_ce_batch, dim3(1), dim3(64), 0, st, part, B, out);
}

template <class T>
static void colsum_of(hipStream_t st, const T* X, const int* starts, int B, int S, int n, double mult, void* ws,
                      double2* out) {
  if (n <= 0 || B <= 0) return;
  MITOK_LAUNCH(k_seq_colsum<T>, dim3((unsigned)((n + 63) / 64 * (long)B)), dim3(256), 0, st, X, starts, S, n, (T*)ws);
  MITOK_LAUNCH(k_seq_sum<T>, dim3((n + 255) / 256), dim3(256), 0, st, (const T*)ws, B, n, mult, out);
}
void colsum(hipStream_t st, const double2* X, int B, int S, int n, double mult, double2* ws, double2* out) {
  colsum_of(st, X, nullptr, B, S, n, mult, ws, out);
}
void colsum_packed(hipStream_t st, const double* X, const int* starts, int B, int n, double2* ws, double2* out) {
  colsum_of(st, X, starts, B, 0, n, 1.0, ws, out);
}

void linear_update(hipStream_t st, double2* W, const double2* dW, double2* mW, double2* vW, long n, double2* b,
                   const double2* db, double2* mb, double2* vb, int V, const TrainStep& ts) {
  const long work = std::max<long>(n, V);
  if (work > 0)
    MITOK_LAUNCH(k_linear_update, dim3((unsigned)((work + 255) / 256)), dim3(256), 0, st, W, dW, mW, vW, n, b, db, mb,
                 vb, V, ts);
}

// ---------------------------------------------------------------------------
// the rest of backward's reverse walk (transformer_network.rs:506-636)
// ---------------------------------------------------------------------------

// sum over a 256-thread block through LDS; every thread gets the total
__device__ double2 block_sum2(double2 v, double2* sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] = cadd(sh[threadIdx.x], sh[threadIdx.x + w]);
    __syncthreads();
  }
  const double2 r = sh[0];
  __syncthreads();
  return r;
}
// f64 / Complex
__device__ __forceinline__ double2 rdivc(double a, double2 z) {
  const double ns = z.x * z.x + z.y * z.y;
  return make_double2(a * z.x / ns, -a * z.y / ns);
}

// NormalNormLayer::backward, Complex arm (norm_layer.rs:132-209), one block per
// row.  The row's input is x, or Re(x + resid) + 0i for the Norm inside a
// SelfAttention layer (add_matrix_3d_c); its forward (normalize, :64-82) is
// recomputed for x_hat, mean and variance.  The reference's f-loop is
// collapsed: with t_d = x_d - mu and the row sums P = sum dout_d t_d,
// D = sum dout_d, M = sum -2 t_d / n, element f's gradient is
//   g_f = dout_f gamma_f / sqrt(v) + gamma_f P (-1/2) v^-3/2 (2 t_f / n)
//         + (-D gamma_f / sqrt(v) + gamma_f P (-1/2) v^-3/2 M) / n,
// v = variance + 1e-8, and the row's input gradient is Re(g_j + (sum_f g_f) dout_j).
// pg[r][j] = dout_j x_hat_j feeds gamma's gradient (n copies per row).
__global__ __launch_bounds__(256) void k_norm_backward(const double2* __restrict__ x, const double2* __restrict__ resid,
                                                       int n, double eps, const double2* __restrict__ gamma,
                                                       const double2* __restrict__ beta,
                                                       const double2* __restrict__ dout, double2* __restrict__ dx,
                                                       double2* __restrict__ pg) {
  __shared__ double2 sh[256];
  const long r = blockIdx.x;
  const double2* xr = x + r * n;
  const double2* gr = dout + r * n;
  const double len = (double)n;
  auto xin = [&](int j) {
    if (!resid) return xr[j];
    return make_double2(xr[j].x + resid[r * n + j].x, 0.0);
  };
  double2 s = make_double2(0.0, 0.0);
  for (int j = threadIdx.x; j < n; j += 256) s = cadd(s, xin(j));
  const double2 mu = cunscale(block_sum2(s, sh), len);
  s = make_double2(0.0, 0.0);
  for (int j = threadIdx.x; j < n; j += 256) {
    const double2 t = csub(xin(j), mu);
    s = cadd(s, cmul(t, t));
  }
  const double2 var = cunscale(block_sum2(s, sh), len);
  const double2 sd = csqrt_nc(cadd(var, make_double2(eps, 0.0)));
  const double2 vb = cadd(var, make_double2(1e-8, 0.0));
  const double2 vroot = csqrt_nc(vb);
  const double2 std_inv = rdivc(1.0, vroot);
  const double2 vpm32 = rdivc(1.0, cmul(vb, vroot));  // powf(1.5) of the principal branch
  double2 P = make_double2(0.0, 0.0), D = P, M = P;
  for (int j = threadIdx.x; j < n; j += 256) {
    const double2 t = csub(xin(j), mu);
    P = cadd(P, cmul(gr[j], t));
    D = cadd(D, gr[j]);
    M = cadd(M, cunscale(cscale(t, -2.0), len));
  }
  P = block_sum2(P, sh);
  D = block_sum2(D, sh);
  M = block_sum2(M, sh);
  const double2 dmu_sum = cmul(D, make_double2(-std_inv.x, -std_inv.y));
  const double2 pv = cmul(cscale(P, -0.5), vpm32);
  double2 gs = make_double2(0.0, 0.0);
  for (int j = threadIdx.x; j < n; j += 256) {
    const double2 t = csub(xin(j), mu);
    const double2 dvar = cmul(gamma[j], pv);
    const double2 dmu = cadd(cmul(dmu_sum, gamma[j]), cmul(dvar, M));
    const double2 g = cadd(cadd(cmul(cmul(gr[j], gamma[j]), std_inv), cmul(dvar, cunscale(cscale(t, 2.0), len))),
                           cunscale(dmu, len));
    gs = cadd(gs, g);
    dx[r * n + j] = g;  // held until the row total is known
    const double2 xh = cadd(cmul(cdiv(t, sd), gamma[j]), beta[j]);
    pg[r * n + j] = cmul(gr[j], make_double2(xh.x, 0.0));
  }
  gs = block_sum2(gs, sh);
  for (int j = threadIdx.x; j < n; j += 256) {
    const double2 g = dx[r * n + j];
    dx[r * n + j] = make_double2(g.x + cmul(gs, gr[j]).x, 0.0);
  }
}


// The attention weights and their gradient from two products' results, one
// wave per query row of a head: A holds Re(q.k) (masked_attention_head.rs:
// 184-205: scaled, plus Re(bias_pos), the causal mask) and becomes
// softmax_complex_padding_real's weights s; dA holds r = Re(dl_ds), dl_ds = G
// conj(V)^T, and becomes backpropagate_softmax_masked_real over the row
// Jacobian s_j (delta_jk - s_k) (utils/derivative.rs:100-131, 253-272):
// dA_j = s_j (r_j - sum_k s_k r_k).  Padded rows 0.  NPL values of a row per
// lane, so both arrays are read and written once.  With the products on the
// matrix cores (8 x 8 heads of 128 rows): 10 us beside 26 us of products, where
// one block per row formed its own dot products in 97.
template <int NPL>
__global__ __launch_bounds__(256) void k_attn_probs_grad(double* __restrict__ A, double* __restrict__ dA,
                                                         const double* __restrict__ bias_re, int mc,
                                                         const uint32_t* __restrict__ mask, long rows, int S, int H,
                                                         double c) {
  const int lane = threadIdx.x & 63;
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int i = (int)(row % S), h = (int)(row / S % H);
  const long b = row / S / H;
  double* a = A + row * S;
  double* g = dA + row * S;
  if (mask[b * S + i] == 0) {
    for (int j = lane; j < S; j += 64) a[j] = g[j] = 0.0;
    return;
  }
  const double* bp = bias_re + ((long)h * mc + i) * mc;
  double sc[NPL], rr[NPL];
  double mx = -INFINITY;
#pragma unroll
  for (int t = 0; t < NPL; ++t) {
    const int j = lane + 64 * t;
    sc[t] = -INFINITY, rr[t] = 0.0;
    if (j < S) {
      sc[t] = j > i ? -1e12 : a[j] * c + bp[j];
      rr[t] = g[j];
    }
    mx = fmax(mx, sc[t]);
  }
  mx = wave_max(mx);
  double sum = 0.0;
#pragma unroll
  for (int t = 0; t < NPL; ++t)
    if (lane + 64 * t < S) {
      sc[t] = exp(sc[t] - mx);
      sum += sc[t];
    }
  sum = wave_sum(sum);
  double sr = 0.0;
#pragma unroll
  for (int t = 0; t < NPL; ++t)
    if (lane + 64 * t < S) {
      sc[t] = sc[t] / sum;
      sr += sc[t] * rr[t];
    }
  sr = wave_sum(sr);
#pragma unroll
  for (int t = 0; t < NPL; ++t) {
    const int j = lane + 64 * t;
    if (j < S) {
      a[j] = sc[t];
      g[j] = sc[t] * (rr[t] - sr);
    }
  }
}

// bias_pos's update on its S x S slice (masked_attention_head.rs:387-393,
// 427-434): the gradient dl_da summed over the sequences (group_gradient_batch),
// clipped; the first update descends, later ones run AdamW from zero moments
// (the reference never reloads prev_m/v_bias_pos).  Only Re(bias_pos) reaches
// the scores, and its update does not depend on the imaginary part.
__global__ __launch_bounds__(256) void k_attn_bias_update(double* __restrict__ bias_re, int mc,
                                                          const double* __restrict__ dA, int B, int H, int S,
                                                          TrainStep ts) {
  const long t = (long)blockIdx.x * 256 + threadIdx.x;
  if (t >= (long)H * S * S) return;
  const int j = (int)(t % S), i = (int)((t / S) % S), h = (int)(t / ((long)S * S));
  double g = 0.0;
  for (int b = 0; b < B; ++b) g += dA[(((long)b * H + h) * S + i) * S + j];
  double* w = bias_re + ((long)h * mc + i) * mc + j;
  double2 m0 = make_double2(0.0, 0.0), v0 = m0;
  *w = update1(make_double2(*w, 0.0), make_double2(g, 0.0), &m0, &v0, ts, true).x;
}

// one parameter array: update1 on every element
__global__ __launch_bounds__(256) void k_param_update(double2* __restrict__ w, const double2* __restrict__ g,
                                                      double2* __restrict__ m, double2* __restrict__ v, long n,
                                                      int weight, TrainStep ts) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) w[i] = update1(w[i], g[i], &m[i], &v[i], ts, weight != 0);
}

// PositionalEncodingLayer::backward (positional_encoding_layer.rs:101-144):
// the pairs of row s rotated back by the forward's angle at position s
// (cs: the forward's (cos, sin) table)
__global__ __launch_bounds__(256) void k_rope_backward(const double2* __restrict__ G, long rows, int S, int d,
                                                       const double2* __restrict__ cs, double2* __restrict__ out) {
  const long t = (long)blockIdx.x * 256 + threadIdx.x;
  const int half = d / 2;
  if (t >= rows * half) return;
  const long r = t / half;
  const int i = (int)(t % half);
  const int pos = (int)(r % S);
  const double2 w = cs[(long)pos * half + i];  // (cos, sin)
  const double2 ge = G[r * d + 2 * i], go = G[r * d + 2 * i + 1];
  out[r * d + 2 * i] = make_double2(ge.x * w.x + go.x * w.y, ge.y * w.x + go.y * w.y);
  out[r * d + 2 * i + 1] = make_double2(-ge.x * w.y + go.x * w.x, -ge.y * w.y + go.y * w.x);
}

// EmbeddingLayer::update_parameters (embedding_layer.rs:223-264): one block
// per distinct target id, its occurrences in the reference's order: the row
// moves by lr * clip(g) / (B V) (g: the gradient row at the target's index),
// then is normalized (utils/normalization.rs:3-20).  A non-finite gradient or
// row raises the error word (the reference panics).
__global__ __launch_bounds__(256) void k_embedding_update(double2* __restrict__ table, int d,
                                                          const uint32_t* __restrict__ ids,
                                                          const int* __restrict__ start, const int* __restrict__ occ,
                                                          const double2* __restrict__ G, double lr, double bs,
                                                          uint32_t* __restrict__ err) {
  __shared__ double2 sh[256];
  double2* row = table + (long)ids[blockIdx.x] * d;
  const double len = (double)d;
  bool bad = false;
  for (int k = start[blockIdx.x]; k < start[blockIdx.x + 1]; ++k) {
    const double2* g = G + (long)occ[k] * d;
    double2 s = make_double2(0.0, 0.0);
    for (int j = threadIdx.x; j < d; j += 256) {
      double2 gj = g[j];
      const double gn = hypot(gj.x, gj.y);
      if (gn > 1.0) gj = cscale(gj, 1.0 / gn);
      if (!(isfinite(gj.x) && isfinite(gj.y))) bad = true;
      const double2 w = csub(row[j], cscale(cunscale(gj, bs), lr));
      if (!(isfinite(w.x) && isfinite(w.y))) bad = true;
      row[j] = w;
      s = cadd(s, w);
    }
    __syncthreads();
    const double2 mean = cunscale(block_sum2(s, sh), len);
    s = make_double2(0.0, 0.0);
    for (int j = threadIdx.x; j < d; j += 256) {
      const double2 t = csub(row[j], mean);
      s = cadd(s, cmul(t, t));
    }
    const double2 sd = csqrt_nc(cadd(cunscale(block_sum2(s, sh), len), make_double2(0.00000000001, 0.0)));
    for (int j = threadIdx.x; j < d; j += 256) row[j] = cdiv(csub(row[j], mean), sd);
    __syncthreads();
  }
  if (bad) atomicOr(err, (uint32_t)EB_TRAIN_NONFINITE);
}

void norm_backward(hipStream_t st, const double2* x, const double2* resid, long rows, int n, double eps,
                   const double2* gamma, const double2* beta, const double2* dout, double2* dx, double2* pg) {
  if (rows > 0) MITOK_LAUNCH(k_norm_backward, dim3((unsigned)rows), dim3(256), 0, st, x, resid, n, eps, gamma, beta, dout, dx, pg);
}

void attn_probs_grad(hipStream_t st, double* A, double* dA, const double* bias_re, int mc, const uint32_t* mask, int B,
                     int S, int H, double c) {
  const long rows = (long)B * H * S;
  const dim3 grid((unsigned)((rows + 3) / 4)), blk(256);
  if (rows <= 0) return;
  if (S <= 64 * 2) MITOK_LAUNCH(k_attn_probs_grad<2>, grid, blk, 0, st, A, dA, bias_re, mc, mask, rows, S, H, c);
  else if (S <= 64 * 8) MITOK_LAUNCH(k_attn_probs_grad<8>, grid, blk, 0, st, A, dA, bias_re, mc, mask, rows, S, H, c);
  else MITOK_LAUNCH(k_attn_probs_grad<48>, grid, blk, 0, st, A, dA, bias_re, mc, mask, rows, S, H, c);  // S <= 3072
}

void attn_bias_update(hipStream_t st, double* bias_re, int mc, const double* dA, int B, int H, int S, const TrainStep& ts) {
  const long total = (long)H * S * S;
  if (total > 0)
    MITOK_LAUNCH(k_attn_bias_update, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, bias_re, mc, dA, B, H, S, ts);
}

void param_update(hipStream_t st, double2* w, const double2* g, double2* m, double2* v, long n, bool weight,
                  const TrainStep& ts) {
  if (n > 0)
    MITOK_LAUNCH(k_param_update, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, w, g, m, v, n, weight ? 1 : 0, ts);
}

void rope_backward(hipStream_t st, const double2* G, long rows, int S, int d, const double2* cs, double2* out) {
  const long total = rows * (d / 2);
  if (total > 0)
    MITOK_LAUNCH(k_rope_backward, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, G, rows, S, d, cs, out);
}

void embedding_update(hipStream_t st, double2* table, int d, const uint32_t* ids, int n_ids, const int* start,
                      const int* occ, const double2* G, double lr, double bs, uint32_t* err) {
  if (n_ids > 0)
    MITOK_LAUNCH(k_embedding_update, dim3(n_ids), dim3(256), 0, st, table, d, ids, start, occ, G, lr, bs, err);
}

// DiscreteWaveletLayer::backward, partial mode (wavelet_discrete_layer.rs:
// 163-207): input row r of sequence b gets sum_k w[r][k] G[b][src[r][k]]
// (four taps at most, src -1: none).  The host builds the table from
// decompress_partial (grad_dwt_1d_trend, dwt.rs:272-282: the low-pass filter
// transposed over the compressed rows), align_gradient_rows_complex (:318-346)
// and the target rows, whose gradient passes through (weight 1).
__global__ __launch_bounds__(256) void k_dwt_backward(const double2* __restrict__ G, int B, int S2, int Sin, int d,
                                                      const int* __restrict__ src, const double* __restrict__ w,
                                                      double2* __restrict__ out) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)B * Sin * d) return;
  const int c = (int)(i % d);
  const long br = i / d;
  const int r = (int)(br % Sin), b = (int)(br / Sin);
  double2 v = make_double2(0.0, 0.0);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int s = src[r * 4 + k];
    if (s >= 0) v = cadd(v, cscale(G[((long)b * S2 + s) * d + c], w[r * 4 + k]));
  }
  out[i] = v;
}

void dwt_backward(hipStream_t st, const double2* G, int B, int S2, int Sin, int d, const int* src, const double* w,
                  double2* out) {
  const long n = (long)B * Sin * d;
  if (n > 0) MITOK_LAUNCH(k_dwt_backward, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, G, B, S2, Sin, d, src, w, out);
}

}  // namespace mitok
