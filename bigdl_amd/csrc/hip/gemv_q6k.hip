// y[M,N] = f(x[M,K] . dequant(W)[N,K]^T) for 1 - 4 rows and a q6_k weight in its checkpoint blocks (210 bytes for 256 codes).
//
// The blocks are read where they lie, a wavefront a weight row, four blocks (840 contiguous bytes) at a time.  A lane owns 16
// codes of a block half: two dwords of low bits, one of high bits, the half's eight scales and the block's scale, requested
// up to eight quads ahead of the arithmetic.  The tile kernel (gemm_rows_kernel.h) reads 64-byte pieces of 16 rows and
// needs a second load for each to shift it into place: it is bound by the number of its requests.  Here it is the
// weight's bytes (head: 3.2 TB/s) and the latency of a first pass (down: one row a wavefront).  Codes and x meet as fp16 in fp32 multiply-adds
// (both exact), the scales are applied in fp32.
#include "gemm_rows_kernel.h"
#include "gemm_rows.h"

namespace bigdl {

constexpr int Q6K_NW = 8;             // wavefronts per workgroup, two workgroups a CU
constexpr int Q6K_U = 4;              // block quadruples of one request group; two groups are in flight
typedef uint32_t q6k_u32 __attribute__((aligned(2)));
typedef uint2v q6k_u64 __attribute__((aligned(2)));

struct Q6kPiece { uint32_t l0, l1, h; uint2v sc; _Float16 d; };

// x in LDS: [M][quads][j = 4][block, half = 8][32 elements], so that the lanes of one read (fixed j) are contiguous
template <int M>
__global__ __launch_bounds__(Q6K_NW * 64, 4) void gemv_q6k_kernel(RowsArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nblk = a.K >> 8, quads = (nblk + 3) >> 2, groups = (quads + Q6K_U - 1) / Q6K_U;
  const int blk = lane >> 4, half = (lane >> 3) & 1, i = lane & 7;
  const int rstride = gridDim.x * Q6K_NW, row0 = blockIdx.x * Q6K_NW + wave;
  const int items = row0 < a.N ? ((a.N - row0 + rstride - 1) / rstride) * groups : 0;

  // request of one item = the quads [4 g, 4 g + 4) of one row; a block past the row's end re-reads the last one
  auto request = [&](Q6kPiece (&p)[Q6K_U], int row, int g) {
    const uint8_t* base = (const uint8_t*)a.w + (int64_t)min(row, a.N - 1) * (nblk * 210);
#pragma unroll
    for (int u = 0; u < Q6K_U; ++u) {
      const uint8_t* b = base + min((g * Q6K_U + u) * 4 + blk, nblk - 1) * 210;
      p[u].l0 = *(const q6k_u32*)(b + 64 * half + 4 * i);
      p[u].l1 = *(const q6k_u32*)(b + 64 * half + 32 + 4 * i);
      p[u].h = *(const q6k_u32*)(b + 128 + 32 * half + 4 * i);
      p[u].sc = *(const q6k_u64*)(b + 192 + 8 * half);
      p[u].d = *(const _Float16*)(b + 208);
    }
    rows_issued();
  };
  Q6kPiece pa[Q6K_U], pb[Q6K_U];
  int row = row0, g = 0;                             // of the item requested last
  auto advance = [&]() { if (++g == groups) { g = 0; row += rstride; } };
  request(pa, row, g);

  for (int m = 0; m < M; ++m) {
    const _Float16* src = a.x + (int64_t)m * a.ldx;
    for (int p = threadIdx.x; p < quads * 128; p += Q6K_NW * 64) {
      const int e = p * 8;
      uint4v v = {0, 0, 0, 0};
      if (e < a.K) v = *(const uint4v*)(src + e);
      const int dst = (m * quads + (e >> 10)) * 1024 + ((e >> 5) & 3) * 256 + ((e >> 7) & 7) * 32 + (e & 31);
      *(uint4v*)((_Float16*)smem + dst) = v;
    }
  }
  __syncthreads();

  float acc[M];
#pragma unroll
  for (int m = 0; m < M; ++m) acc[m] = 0.0f;
  auto work = [&](const Q6kPiece (&p)[Q6K_U], int wrow, int wg) {
#pragma unroll
    for (int u = 0; u < Q6K_U; ++u) {
      const int quad = wg * Q6K_U + u;
      if (quad >= quads) break;
      float part[M];
#pragma unroll
      for (int m = 0; m < M; ++m) part[m] = 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // codes 32 j + 4 i .. + 3 of the half: low bits from dword j & 1, nibble j >> 1; high bits 2 j, 2 j + 1
        const uint32_t code = (((j & 1 ? p[u].l1 : p[u].l0) >> (4 * (j >> 1))) & 0x0F0F0F0Fu) | (((p[u].h >> (2 * j)) & 0x03030303u) << 4);
        const half2v off = {(_Float16)1056.0f, (_Float16)1056.0f};       // 1024 + 32
        const half2v c0 = u2h(__builtin_amdgcn_perm(0x64646464u, code, 0x04010400u)) - off;
        const half2v c1 = u2h(__builtin_amdgcn_perm(0x64646464u, code, 0x04030402u)) - off;
        const float s = (float)(int8_t)(p[u].sc[j >> 1] >> (16 * (j & 1) + 8 * (i >> 2)));
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const half4 xv = *(const half4*)((const _Float16*)smem + (m * quads + quad) * 1024 + j * 256 + lane * 4);
          float dot = (float)c0[0] * (float)xv[0];
          dot = fmaf((float)c0[1], (float)xv[1], dot);
          dot = fmaf((float)c1[0], (float)xv[2], dot);
          dot = fmaf((float)c1[1], (float)xv[3], dot);
          part[m] = fmaf(s, dot, part[m]);
        }
      }
      const float d = quad * 4 + blk < nblk ? (float)p[u].d : 0.0f;
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = fmaf(d, part[m], acc[m]);
    }
    if (wg != groups - 1) return;
    float y = 0.0f;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      float v = acc[m];
      acc[m] = 0.0f;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
      if (lane == m) y = v;
    }
    if (lane < M) {
      if (a.bias != nullptr) y += (float)((const _Float16*)a.bias)[wrow];
      y = act_apply(a.act, y);
      const int64_t oi = (int64_t)lane * a.ldo + wrow;
      if (a.out_type == OUT_F16) {
        if (a.residual) y += load_out<OUT_F16>(a.residual, oi);
        store_out<OUT_F16>(a.out, oi, y);
      } else if (a.out_type == OUT_BF16) {
        if (a.residual) y += load_out<OUT_BF16>(a.residual, oi);
        store_out<OUT_BF16>(a.out, oi, y);
      } else {
        if (a.residual) y += load_out<OUT_F32>(a.residual, oi);
        store_out<OUT_F32>(a.out, oi, y);
      }
    }
  };
  // (requests are never under a condition: that would cost the counts of the waits.  Past the last item they re-read a row.)
  for (int it = 0; it < items; it += 2) {
    const int row_a = row, g_a = g;
    advance();
    const int row_b = row, g_b = g;
    request(pb, row_b, g_b);
    work(pa, row_a, g_a);
    advance();
    request(pa, row, g);
    if (it + 1 < items) work(pb, row_b, g_b);
  }
}

static size_t q6k_lds(int M, int K) { return (size_t)M * ((K / 256 + 3) / 4) * 2048; }

// Time against the tile kernel's best tiling, us: 1 / 2 / 3 / 4 rows, 4096 x 11008 16.9 / 18.1 / 21.1 / 25 against 24.8 - 25.1;
// 12288 x 4096 17.2 / 19.4 / 21.8 / 24.1 against 27.2 - 28.0; 32000 x 4096 33 / 38 / 44 / 50 against 58 - 60; 2048 x 2048 5.3 - 7.0
// against 12.6 - 13.3.  Every further row costs 2 - 6 us, so four are the limit; two workgroups' x have to fit a CU's LDS.
bool gemv_q6k_takes(const RowsArgs& a) {
  return a.M <= 4 && a.gamma == nullptr && a.splitk <= 1 && q6k_lds(a.M, a.K) <= 80 * 1024;
}

template <int M>
static int launch(const RowsArgs& a, hipStream_t st) {
  const size_t lds = q6k_lds(M, a.K);
  if (!gemv_allow_lds((const void*)gemv_q6k_kernel<M>, 80 * 1024)) return -101;
  const int need = (a.N + Q6K_NW - 1) / Q6K_NW, most = 2 * gemv_cu_count();
  hipLaunchKernelGGL(gemv_q6k_kernel<M>, dim3(need < most ? need : most), dim3(Q6K_NW * 64), lds, st, a);
  return HIP_CHECK_LAUNCH();
}
int gemv_q6k_launch(const RowsArgs& a, hipStream_t st) {
  switch (a.M) {
    case 1: return launch<1>(a, st);
    case 2: return launch<2>(a, st);
    case 3: return launch<3>(a, st);
    default: return launch<4>(a, st);
  }
}
}  // namespace bigdl
