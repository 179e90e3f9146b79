// train.hpp — launch wrappers of training: the tiled MFMA product with its
// operand forms (gemm_mfma.hip, also the prompt pass's), the softmax rows
// (kernels.hip) and backward's kernels (train.hip).  Apart from kernels.hpp,
// which the resident loop's kernels are built on.
#pragma once

#include "kernels.hpp"

namespace mitok {

// ---- MFMA-tiled product (gemm_mfma.hip): block tile GBM x GBN, K step GBK ----
constexpr int GBM = 64, GBN = 64, GBK = 8;
// the first `whole` output tiles are one block each, the `rest` P blocks of kchunk of K
struct MfmaPlan {
  int whole = 0, rest = 0, P = 1, kchunk = 0;
  long blocks() const { return whole + (long)rest * P; }
  size_t ws_bytes() const { return P > 1 ? (size_t)rest * P * GBM * GBN * sizeof(double2) : 0; }
};
// How an operand is read: OP_T the transpose of the stored row-major array,
// OP_CJ its conjugate, OP_RE its imaginary parts are zero, OP_F64 it is stored
// as doubles.
constexpr int OP_T = 1, OP_CJ = 2, OP_RE = 4, OP_F64 = 8, OP_H = OP_T | OP_CJ;
struct GemmOpnd {
  const void* p = nullptr;
  long ld = 0;
  int flags = 0;
};
// `n` independent products of one shape: product z's operands and output
// (elements of each array's own type) start at (z / inner) * outer step + (z %
// inner) * inner step; the result is multiplied by `scale` (EPI_STORE)
struct MfmaBatch {
  int n = 1, inner = 1;
  long a0 = 0, a1 = 0, b0 = 0, b1 = 0, c0 = 0, c1 = 0;
  double scale = 1.0;
  // a real A: the row a zero row of A would give, [N], zeros before the launch;
  // NaN is left where B's column holds an infinity or NaN
  double2* zero_row = nullptr;
};
// ERR_ARG for a combination of mode and operand forms nothing uses
int launch_zgemm_mfma(hipStream_t st, const MfmaPlan& p, const GemmOpnd& A, const GemmOpnd& B, int M, int N, int K,
                      const Epi& ep, const Argmax& am, double2* ws, uint32_t* cnt, const MfmaBatch& bt = MfmaBatch());
// the tiled product for any M, with its plan's split workspace (gemm.hip)
size_t gemm_tiled_ws_bytes(int M, int N, int K);
int gemm_tiled(hipStream_t st, int M, int N, int K, const GemmOpnd& A, const GemmOpnd& B, const Epi& ep, const Sync& sy,
               const MfmaBatch& bt = MfmaBatch());

// x [rows][V]: real logits in, probabilities out
void softmax_rows(hipStream_t st, double* x, int rows, int S, int V, const uint32_t* row_mask, int mode);

// ---- the output head's training step (train.hip) ----
struct TrainStep {
  int first = 0;      // the first update: clipped gradient descent (linear_layer.rs:159-174)
  double lr = 0.0;    // the layer's learning rate
  double batch = 1;   // sequences in the batch (the descent divides by it)
  int time_step = 0;  // AdamW's bias-correction step (at least 1)
};
// packed softmax gradient G [n][V]: row i = (P[r][c] - [c == tgt[r]]) / norm[r / S] of r = rows[i], zeros for r < 0
void softmax_grad(hipStream_t st, const double* P, int n, int V, const int* rows, const int* tgt, const double* norm,
                  int S, double* G);
// out[packed[r]] = X[r]; the rows of packed row `zero` leave zeros there, NaN where one of them is not finite
void pack_rows(hipStream_t st, const double2* X, long rows, int d, const int* packed, int zero, double2* out);
// out[r] = in[packed[r]]
void unpack_rows(hipStream_t st, const double2* in, long rows, int d, const int* packed, double2* out);
// cross_entropy_loss_batch of P [B][S][V] for targets [B][T] (tlen[b] each):
// part [B] the sequences' losses, out [2] the batch loss (re, im); T <= CE_MAX_T
constexpr int CE_MAX_T = 8192;
void cross_entropy(hipStream_t st, const double* P, int B, int S, int V, const uint32_t* tgt, const uint32_t* tlen,
                   int T, double* part, double* out);
// G = mask[r] ? dH * conj(GELU'(Z)) : 0 (layer.rs:181-192, derivative.rs:48-84); mask may be null (all rows)
void gelu_backward(hipStream_t st, const double2* dH, const double2* Z, const uint32_t* mask, long rows, int F,
                   double2* G);
// W [n], b [V] updated in place from dW, db (moments mW, vW, mb, vb)
void linear_update(hipStream_t st, double2* W, const double2* dW, double2* mW, double2* vW, long n, double2* b,
                   const double2* db, double2* mb, double2* vb, int V, const TrainStep& ts);
// the Norm's backward per row of x (or Re(x + resid) + 0i); dx real rows, pg = dout * x_hat
void norm_backward(hipStream_t st, const double2* x, const double2* resid, long rows, int n, double eps,
                   const double2* gamma, const double2* beta, const double2* dout, double2* dx, double2* pg);
// out[j] = mult * sum over sequences b of the row sum of X[b][:][j] (four runs of rows, each in order, then the
// sequences in order); ws [B][n]
void colsum(hipStream_t st, const double2* X, int B, int S, int n, double mult, double2* ws, double2* out);
// the same of packed real rows, sequence b's at [starts[b], starts[b + 1])
void colsum_packed(hipStream_t st, const double* X, const int* starts, int B, int n, double2* ws, double2* out);
// A [B][H][S][S]: Re(q.k) in, attention weights out; dA: Re(G conj(V)^T) in, dl_da out (S <= 3072)
void attn_probs_grad(hipStream_t st, double* A, double* dA, const double* bias_re, int mc, const uint32_t* mask, int B,
                     int S, int H, double c);
// Re(bias_pos)[h][:S][:S] updated from dA summed over the batch (zero moments each call)
void attn_bias_update(hipStream_t st, double* bias_re, int mc, const double* dA, int B, int H, int S,
                      const TrainStep& ts);
// w [n] updated in place (weight: AdamW's EPSILON floor on v_hat's norm)
void param_update(hipStream_t st, double2* w, const double2* g, double2* m, double2* v, long n, bool weight,
                  const TrainStep& ts);
// RoPE's backward on rows [rows][d] of sequences of S rows (cs: the forward's table)
void rope_backward(hipStream_t st, const double2* G, long rows, int S, int d, const double2* cs, double2* out);
// the wavelet layer's backward: out [B][Sin][d] from G [B][S2][d] through a tap table [Sin][4]
void dwt_backward(hipStream_t st, const double2* G, int B, int S2, int Sin, int d, const int* src, const double* w,
                  double2* out);
// the embedding rows of n_ids distinct ids, each with occurrences occ[start[u] .. start[u+1]) (rows of G)
void embedding_update(hipStream_t st, double2* table, int d, const uint32_t* ids, int n_ids, const int* start,
                      const int* occ, const double2* G, double lr, double bs, uint32_t* err);

}  // namespace mitok
