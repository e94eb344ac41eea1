// The decayed outer-product rule of time mixing, row by row and in chunks of 64 tokens on the matrix cores (gated_rule.h's kernels,
// RULE_BONUS): per head a state S [D, D],
//
//   y = (S + diag(u) k v')' q,   S = diag(f) S + k v',   f = exp(-exp(z + b))
//   out = y / sqrt(mean(y^2) + eps) * gain * silu(g)
//
// with the decays, the heads' norm and the gate, which the walk of recurrent.hip has around it as kernels of their own.  In chunks, bound by
// the exponentials and the matrix products of the scores: 2,048 tokens, 32 heads of 64 (us), the walk 952 and 27 around it, in chunks 138
// (118 with decays as differences of sums and scores in 32 bits: the error of the read-outs was 1.9 times the walk's at moderate decays and 32
// times where hard ones stand among gentle ones, the state's 1.2 and 100 times; now 0.9 and 0.8, 0.9 and 1.0).  Row by row, bound by the chain of a row: 8 requests of one token, 32 heads of 64, the walk
// 8.3 and 7.4 around it, here 8.2.
#include "gated_rule.h"

namespace {
RuleArgs outer_rule(const void* rows, long ld, int off_k, int off_v, int off_g, const float* z, const float* bias, const float* bonus,
                    const float* gain, float eps, float* state, long slot_stride, const int* cu, const int* slot, void* out, int H, int D) {
  RuleArgs a{};
  a.raw = rows; a.ld = ld; a.off_q = 0; a.off_k = off_k; a.off_v = off_v; a.off_g = off_g;
  a.z = z; a.bias = bias; a.bonus = bonus; a.gain = gain; a.gain_stride = D; a.eps = eps;
  a.state = state; a.slot_stride = slot_stride; a.cu = cu; a.slot = slot; a.out = out; a.H = H; a.D = D; a.V = D;
  return a;
}
int check(const char* what, const RuleArgs& a, int dtype, int n_req) {
  GIBBS_REQUIRE(a.raw && a.z && a.bias && a.bonus && a.gain && a.state && a.slot && a.out, "%s: null operand", what);
  GIBBS_REQUIRE(n_req > 0 && a.H > 0 && a.H <= 65535 && a.D > 0 && a.ld >= (long)a.H * a.D && a.off_k >= 0 && a.off_v >= 0 && a.off_g >= 0 &&
                    a.slot_stride >= (long)a.H * a.D * a.D, "%s: requests=%d heads=%d D=%d", what, n_req, a.H, a.D);
  GIBBS_REQUIRE(dtype == GIBBS_F32 || dtype == GIBBS_BF16, "%s: unknown dtype %d", what, dtype);
  return 0;
}
}  // namespace

// Whether the row kernel takes a head's size (a state that is aligned to 16 bytes, or D up to 512).
GIBBS_EXPORT int gibbs_decayed_outer_rows_take(int D) { return D <= STEP_THREADS && rule_rows_take(D, D); }
// cu null: row n is request n's; else the rows cu[r] .. cu[r + 1].  Operands as below, z by the step's rows.
GIBBS_EXPORT int gibbs_decayed_outer_rows(const void* rows, long ld, int off_k, int off_v, int off_g, const float* z, const float* bias,
                                          const float* bonus, const float* gain, float eps, float* state, long slot_stride, const int* cu,
                                          const int* slot, void* out, int dtype, int n_req, int H, int D, hipStream_t stream) {
  const RuleArgs a = outer_rule(rows, ld, off_k, off_v, off_g, z, bias, bonus, gain, eps, state, slot_stride, cu, slot, out, H, D);
  if (check("decayed_outer_rows", a, dtype, n_req)) return 1;
  GIBBS_REQUIRE(gibbs_decayed_outer_rows_take(D), "decayed_outer_rows: heads of %d", D);
  if (dtype == GIBBS_F32 ? launch_rule_rows<float, RULE_BONUS>(a, n_req, stream) : launch_rule_rows<bf16, RULE_BONUS>(a, n_req, stream)) return 1;
  GIBBS_LAUNCH_STATUS("decayed_outer_rows");
}

// Whether a head's size is taken, and the floats of workspace that `rows` rows of `n_req` requests need.
GIBBS_EXPORT int gibbs_decayed_outer_chunks_take(int D) { return rule_chunks_take(D, D, RULE_BONUS); }
GIBBS_EXPORT long gibbs_decayed_outer_chunks_workspace(int rows, int n_req, int H, int D) { return rule_chunks_workspace(rows, n_req, H, D, D); }

// The rows cu[0] .. of n_req requests (rows and out are addressed by the step's rows, cu may start above 0), n_rows in all.  q, k, v, g:
// rows of H * D values in one type at `rows` + 0, off_k, off_v, off_g values (row stride ld); z [n_rows, H * D] float32: those rows'
// log rates without the bias; bias, bonus, gain [H * D]; state [slots][H][D][D]; out [.., H * D] in the rows' type.
GIBBS_EXPORT int gibbs_decayed_outer_chunks(const void* rows, long ld, int off_k, int off_v, int off_g, const float* z, const float* bias,
                                            const float* bonus, const float* gain, float eps, float* state, long slot_stride, const int* cu,
                                            const int* slot, void* out, float* workspace, int dtype, int n_rows, int n_req, int H, int D,
                                            hipStream_t stream) {
  const RuleArgs a = outer_rule(rows, ld, off_k, off_v, off_g, z, bias, bonus, gain, eps, state, slot_stride, cu, slot, out, H, D);
  if (check("decayed_outer_chunks", a, dtype, n_req)) return 1;
  GIBBS_REQUIRE(cu && workspace && n_rows > 0 && n_req <= 65535 && gibbs_decayed_outer_chunks_take(D), "decayed_outer_chunks: rows=%d requests=%d, heads of %d", n_rows, n_req, D);
  const int places = ceil_div(n_rows, CHUNK) + n_req;      // (more than the requests' chunks can be)
  if (dtype == GIBBS_F32 ? launch_chunks<float, RULE_BONUS>(a, workspace, places, n_req, stream) : launch_chunks<bf16, RULE_BONUS>(a, workspace, places, n_req, stream)) return 1;
  GIBBS_LAUNCH_STATUS("decayed_outer_chunks");
}
