// A decode step of one row (bf16: up to four) as one resident launch: arguments and host entry points (decode_stream.hip).
#pragma once
#include "../common.h"
#include "../qweight.h"

namespace aios {

// a workgroup's rows of a product, one record a product, in the order of the step (Q | K | V, O, gate/up and down of each
// layer, the head)
struct alignas(16) DsJob {
  int r0, nrows;       // rows of the product's output
  int chunks, slots;   // of 32 weights (bit 30: Q6_K, else Q4_K), or bf16 groups of four rows by 512 columns; of the ring
};
constexpr int DS_Q6 = 1 << 30;
// ... and what its loaders copy: planes of qweight.h at its first row
struct alignas(64) DsCopy {
  const uint8_t* p[4];  // (bf16: the first row, and the bytes of a row)
  DsJob job;
};

// what launches leave each other; all zero before the first one
struct DsCtl {
  unsigned arrive, state, done;  // of the running launch: workgroups there, 1 go / 2 given up, workgroups gone (above 16 bits: that waited too long)
  unsigned epoch;                // numbers of the exchanges used so far
  unsigned failed;               // the last resident launch gave up: the launch behind it does the step
  unsigned alone;                // steps that the launch behind did
};

struct DsArgs {
  const DsCopy* jobs;     // [4 n_layers + 1][parts]
  const float* gains;     // [2 n_layers + 1][d]: of the norms in front of QKV, gate/up, .., the head
  const float* qk_gains;  // [2 n_layers][head_dim] of q and k, or null
  const float* bias;      // [n_layers][rows of QKV], or null
  const float* kv_scale;  // [2 n_layers] of K and V (fp8 caches)
  uint8_t *kc, *vc;       // the cache pools, a layer kv_layer bytes behind the other
  size_t kv_layer;
  int n_layers, d, n_heads, n_kv_heads, ff, vocab, max_ctx, rope_neox, kv_fp8;
  int parts;           // workgroups that the step is dealt to
  int bf16;            // 1: bf16 weights, else Q4_K / Q6_K with int8 activations
  int rows;            // of the batch: 1, bf16 up to 4
  int ring;            // (bf16) slots of the ring
  int bt_stride, ldl;  // of the block tables and the logits of a row
  int row_sums;        // words of the sums of a layer product's rows in LDS, of one buffer
  int own_rows;        // rows of the residual that a workgroup has, at most
  int area_bytes;      // LDS of the staged operand (behind the head's its sums) or of the attention's rows
  float eps, scale;
  const float* x;      // the embedding
  float* logits;
  const float2* rope_cs;
  const int *pos, *blocks;  // positions of the rows, their block tables
  // exchanges, one a layer each, a row of the batch behind the other: the residual behind O and behind down times the next norm's gains, its squares' sum by workgroup, rows of QKV,
  // heads, pairs of gate/up
  uint64_t *xn, *sq, *qkv, *attn, *h;
  float* resid;                        // [rows][d]: the residual, for a launch of one workgroup
  uint64_t* part;                      // results of runs of keys (one for all layers)
  int nqkv;
  DsCtl* ctl;
  unsigned* host_failed;    // pinned: counts steps that the launch behind had to do
  unsigned long long gate_ticks, wait_ticks;  // of 10 ns
  int alone;           // 1: the launch behind, one workgroup that takes all parts in turn
};

constexpr int DS_PMAX = 32;  // runs of keys that a head's attention is split into, at most

// elements of the exchanges
inline size_t ds_part_words(int n_heads, int hd) { return (size_t)n_heads * DS_PMAX * (hd + 2); }  // of one row

// rows [r0, r0 + nrows) of matrix w, whose first row is row row0 of the output
DsCopy ds_job(const QWeight& w, int r0, int nrows, int row0);
// Whether the step of `rows` rows of such a model can run resident: the shapes that the kernel is built for, its LDS (fills rows,
// row_sums, own_rows, area_bytes and ring).  max_sums, head_sums: words of the sums of a workgroup's rows, of a layer's product at most and of
// the head.  Formats, ranks and activations are the caller's to check.
bool ds_plan(DsArgs& a, int head_dim, int max_sums, int head_sums, int rows);
// words of the sums of this many rows of w
int ds_sums(const QWeight& w, int rows);
// the resident launch and the one behind it (which returns at once unless the first gave up)
void launch_decode_stream(const DsArgs& a, int head_dim, hipStream_t st);

}  // namespace aios
