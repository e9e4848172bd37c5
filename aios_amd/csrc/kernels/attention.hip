// Split-K flash-decode GQA attention over the paged KV cache (decode shape),
// with the log-sum-exp combine fused in (last-arriving workgroup per (row, kv-head)).
//
// grid = (roles, 1, B), 512 threads (8 waves).  The context is cut into 32-key tiles, dealt over the
// waves of the P workgroups of a (row, KV head); a wave keeps its own online-softmax state for the KV head's
// query heads (attn_core in attn_decode.h).  Short contexts of small batches: a workgroup per query head, without a
// combine (attn_short).
//
// Combine: with more than one active workgroup each writes its partial (o, m, l) with
// write-through (sc1, agent scope) stores, drains them (s_waitcnt vmcnt(0)), and after a
// workgroup barrier one lane takes an agent-scope ticket for (row, kv head).  The last arriver
// reads every partial's (m, l) in one parallel sweep (one lane per partial), then each thread
// sums its outputs over the partials with independent loads -- the write-through hand-off of
// CDNA guide §6 Guideline 16 / split-K item 2 -- and re-arms the counter.
#include "attn_decode.h"

namespace aios {

// (head_dim 64: two workgroups to a CU, 128 registers; 128: the tiles in flight take the register file)
template <int HD, int G, bool F8>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(HD == 64 ? 4 : 2))) attn_decode_kernel(AttnDecodeArgs a, AttnSplit s) {
  kernarg_warm<sizeof(AttnDecodeArgs) + sizeof(AttnSplit)>();
  attn_role<HD, G, F8>(a, s, blockIdx.x);
}

// a workgroup or more per query head for every context (attn_lanes_only)
template <int HD, bool F8>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) attn_lanes_kernel(AttnDecodeArgs a, AttnSplit s) {
  kernarg_warm<sizeof(AttnDecodeArgs) + sizeof(AttnSplit)>();
  attn_lanes<HD, F8, true>(a, blockIdx.x / s.p, blockIdx.x / s.p, blockIdx.x % s.p, s.p);
}

template <int HD, bool F8>
static void launch_hd(const AttnDecodeArgs& a, int G, hipStream_t st) {
  AttnSplit sp;
  const dim3 grid(attn_plan(a, G, sp), 1, a.B), block(512);
  constexpr int lds = at_lds_bytes<HD>();
  if constexpr (HD == 128) {
    if (attn_lanes_only(a, G)) {
      hipLaunchKernelGGL((attn_lanes_kernel<HD, F8>), dim3(a.n_heads * sp.p, 1, a.B), block, AT_NW * HD * 4, st, a, sp);
      return;
    }
  }
  switch (G) {
    case 1: hipLaunchKernelGGL((attn_decode_kernel<HD, 1, F8>), grid, block, lds, st, a, sp); break;
    case 2: hipLaunchKernelGGL((attn_decode_kernel<HD, 2, F8>), grid, block, lds, st, a, sp); break;
    case 4: hipLaunchKernelGGL((attn_decode_kernel<HD, 4, F8>), grid, block, lds, st, a, sp); break;
    case 5: hipLaunchKernelGGL((attn_decode_kernel<HD, 5, F8>), grid, block, lds, st, a, sp); break;
    case 8: hipLaunchKernelGGL((attn_decode_kernel<HD, 8, F8>), grid, block, lds, st, a, sp); break;
    default: throw std::runtime_error("attn_decode: unsupported GQA group size " + std::to_string(G));
  }
}

// `split` (kept in the args for the API) encodes P * ATTN_CHUNK: the number of workgroups per
// (row, head set) in the long-context mode.  Target one workgroup per CU for the whole grid (a
// 512-thread workgroup of this kernel fills a CU's register file), 1..64 per head set, each
// owning at least one 128-key pass of a max_ctx context.
int attn_decode_split(int max_ctx, int B, int n_kv_heads) {
  const int nch = std::max(1, max_ctx / 128);
  // AIOS_ATTN_WG_PER_CU (default 1): long-context workgroups per CU the split aims for
  const int per_cu = std::max(1, std::min(4, attn_env_int("AIOS_ATTN_WG_PER_CU", 1)));
  const int P = std::max(1, std::min({64, nch, 256 * per_cu / std::max(1, B * n_kv_heads)}));
  return P * ATTN_CHUNK;
}

void launch_attn_decode(const AttnDecodeArgs& a, hipStream_t st) {
  if (a.n_heads % a.n_kv_heads) throw std::runtime_error("attn_decode: n_heads % n_kv_heads != 0");
  if (!a.counters) throw std::runtime_error("attn_decode: counters buffer required ([B][n_heads])");
  if (a.max_ctx % 128) throw std::runtime_error("attn_decode: max_ctx must be a multiple of 128");
  const int G = a.n_heads / a.n_kv_heads;
  const AttnDecodeArgs b = attn_resolve(a);
  if (b.split % ATTN_CHUNK) throw std::runtime_error("attn_decode: split must be a multiple of ATTN_CHUNK");
  if (a.head_dim == 128) {
    if (a.kv_fp8) launch_hd<128, true>(b, G, st);
    else launch_hd<128, false>(b, G, st);
  } else if (a.head_dim == 64) {
    if (a.kv_fp8) launch_hd<64, true>(b, G, st);
    else launch_hd<64, false>(b, G, st);
  } else {
    throw std::runtime_error("attn_decode: head_dim must be 64 or 128");
  }
}

}  // namespace aios
