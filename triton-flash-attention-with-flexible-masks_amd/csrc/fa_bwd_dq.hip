// dQ of the split backward: the kernel and its launch (the work itself is in fa_dq_body.h).
#include "fa_tile.h"

namespace fa {

#ifdef FA_TRACE
// words: 0 start, 1 rows and ids known, 2 before the tile loop, 3 after it, 4 end, 5 key tiles computed, 6 (merging workgroup only) partial result stored and arrival counted, 7 tile | chunk << 16 | chunks << 24 (-1: left at once)
FA_TRACE_ARRAY(g_trace_dq);
#endif

}  // namespace fa
#include "fa_dq_body.h"
namespace fa {

template <typename Tag, int D, bool CAUSAL, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D <= 64 ? 3 : 2, D <= 64 ? 3 : 2)))
void bwd_dq_kernel(const KArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  dq_body<Tag, D, CAUSAL, MODE>(a, (int)blockIdx.x, smem);
}

template <typename Tag, int D, bool CAUSAL, int MODE>
static int launch_one(const KArgs& a, hipStream_t s) {
  constexpr size_t lds = dq_lds<D>();
  auto kern = bwd_dq_kernel<Tag, D, CAUSAL, MODE>;
  static bool lds_allowed[64] = {};   // per kernel instantiation and device
  if (int e = allow_lds(kern, lds, lds_allowed)) return e;
  hipLaunchKernelGGL(kern, dim3(grid_blocks(launch_slots<MODE>(a), launch_groups<MODE>(a))), dim3(256), lds, s, a);
  return (int)hipGetLastError();
}

template <typename Tag, int D>
static int launch_cd(const KArgs& a, bool causal, bool doc, hipStream_t s) {
  if (doc) return causal ? launch_one<Tag, D, true, GEO_DOC>(a, s) : launch_one<Tag, D, false, GEO_DOC>(a, s);
  if (geo_general(a)) return causal ? launch_one<Tag, D, true, GEO_GENERAL>(a, s) : launch_one<Tag, D, false, GEO_GENERAL>(a, s);
  return causal ? launch_one<Tag, D, true, GEO_PLAIN>(a, s) : launch_one<Tag, D, false, GEO_PLAIN>(a, s);
}

template <typename Tag>
static int launch_d(const KArgs& a, int D, bool causal, bool doc, hipStream_t s) {
  switch (D) {
    case 128: return launch_cd<Tag, 128>(a, causal, doc, s);
    case 64: return launch_cd<Tag, 64>(a, causal, doc, s);
    case 32: return launch_cd<Tag, 32>(a, causal, doc, s);
    case 16: return launch_cd<Tag, 16>(a, causal, doc, s);
    default: return -1;
  }
}

#ifdef FA_TRACE
int trace_read_dq(long long* host, int n) { return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(g_trace_dq), size_t(n) * 8); }
#endif

int launch_bwd_dq(const KArgs& a, int dtype, int D, bool causal, bool doc, hipStream_t s) {
  return dtype == FA_DTYPE_BF16 ? launch_d<bf16_t>(a, D, causal, doc, s) : launch_d<fp16_t>(a, D, causal, doc, s);
}

}  // namespace fa
