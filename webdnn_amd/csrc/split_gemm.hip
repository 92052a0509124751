// Gemm / MatMul on the bf16 matrix cores (split_product.h holds the kernel and says what it computes).
#include "split_product.h"

namespace wdhc {
int launch_split_gemm(bool b_kc, const SplitPlan &s, Params &p, int nz) {
  return b_kc ? launch_split<B_KC>(s, p, nz) : launch_split<B_MC>(s, p, nz);
}

int launch_split_group(bool b_kc, int count, Params *p) {
  GroupParams g;
  long long blocks = 0;
  g.count = count;
  for (int i = 0; i < count; i++) {
    Params &q = p[i];
    q.tiles_m = (q.m + 63) / 64;
    q.tiles_n = (q.n + 63) / 64;
    q.nz = 1;
    q.full_tiles = q.tiles_m * q.tiles_n;
    q.tail_tiles = 0;
    q.tail_split = 1;
    q.kchunk = 0;
    q.fd_tiles_per_z = make_fastdiv(q.full_tiles);
    q.fd_group = make_fastdiv((long long)TILE_GROUP * q.tiles_n);
    q.fd_last_rows = make_fastdiv(q.tiles_m % TILE_GROUP ? q.tiles_m % TILE_GROUP : 1);
    q.fd_tail_tiles = make_fastdiv(1);
    g.first[i] = (int)blocks;
    g.p[i] = q;
    blocks += q.full_tiles;
  }
  g.first[count] = (int)blocks;
  g_last_plan = {64, 64, 1, b_kc ? WDH_FORM_GEMM_KC : WDH_FORM_GEMM_MC, blocks, 0};
  if (b_kc) hipLaunchKernelGGL((split_group_kernel<B_KC, 4>), dim3((unsigned)blocks), dim3(1024), 0, wdh::stream(), g);
  else hipLaunchKernelGGL((split_group_kernel<B_MC, 4>), dim3((unsigned)blocks), dim3(1024), 0, wdh::stream(), g);
  WDH_LAUNCH_CHECK();
  return WDH_OK;
}
}  // namespace wdhc
