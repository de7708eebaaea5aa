// y[M,N] = f(x[M,K] . dequant(W)[N,K]^T) for 1 - 4 rows and a q6_k weight in its checkpoint blocks (210 bytes for 256 codes).
//
// The blocks are read where they lie, a wavefront a weight row, eight blocks (1680 contiguous bytes) at a time: aligned 16-byte
// pieces go straight to the wavefront's own patch of LDS, one item ahead of the arithmetic.  A lane owns 16 codes of a block half:
// two dwords of low bits, one of high bits, four of the half's scales and the block's scale, shifted into place on their way out of
// LDS (a row starts at any even byte).  Requested by the lanes themselves those are five 2-byte-aligned loads a quad of blocks, and
// even without arithmetic and with the weight in the caches they took 11.6 of 16.5 us (4096 x 11008); now 12.0 us, 7.0 of them so.
// Bound by the LDS reads and the vector operations on the codes (3.4 us of the 12.0) and by a short row's first pass.  Codes and x
// meet as fp16 in two-term dot products with fp32 sums (products exact), the scales are applied in fp32.
#include "gemm_rows_kernel.h"
#include "gemm_rows.h"

namespace bigdl {

constexpr int Q6K_U = 2;                             // block quads of one item
constexpr int Q6K_PIECES = (Q6K_U * 840 + 2 + 15) / 16, Q6K_PATCH = Q6K_PIECES * 16;       // of an item, from the dword in front of it
typedef uint2v q6k_u64 __attribute__((aligned(4)));
typedef __attribute__((address_space(3))) void q6k_lds_t;

// x in LDS: [M][quads][j = 4][block, half = 8][32 elements], so that the lanes of one read (fixed j) are contiguous; behind it two patches
// a wavefront.  NW: wavefronts of a workgroup; OCC: wavefronts a SIMD that the registers have to allow
template <int M, int NW, int OCC>
__global__ __launch_bounds__(NW * 64, OCC) void gemv_q6k_kernel(RowsArgs a) {
  constexpr int U = Q6K_U, DMAS = (Q6K_PIECES + 63) / 64;      // of 64 lanes, the last of fewer
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nblk = a.K >> 8, quads = (nblk + 3) >> 2, groups = (quads + U - 1) / U;
  const int blk = lane >> 4, half = (lane >> 3) & 1, i = lane & 7;
  const int rstride = gridDim.x * NW, row0 = blockIdx.x * NW + wave;
  const int items = row0 < a.N ? ((a.N - row0 + rstride - 1) / rstride) * groups : 0;
  char* const patches = smem + M * quads * 2048 + wave * (2 * Q6K_PATCH);
  const int row_bytes = nblk * 210;
  auto row_at = [&](int row) { return (uint64_t)a.w + (int64_t)row * row_bytes; };

  // request of one item = the quads [U g, U g + U) of one row into patch `at`, from the dword that holds their first byte (840 U is a
  // multiple of 16).  The descriptor ends with the dword of the row's last byte and is empty past the last item: what lies behind is
  // not fetched.  (The whole offset is the lane's, so that all of it is held against that end.)
  auto request = [&](int at, int row, int g) {
    const uint64_t w = row_at(row);
    const rows_rsrc wb = rows_buffer((const void*)(w & ~3ull), row < a.N ? (int)(((w & 3) + row_bytes + 3) & ~3u) : 0);
#pragma unroll
    for (int c = 0; c < DMAS; ++c)
      if (c + 1 < DMAS || lane < Q6K_PIECES - 64 * (DMAS - 1))
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wb, (q6k_lds_t*)(patches + at * Q6K_PATCH + c * 1024), 16, lane * 16 + c * 1024 + g * (U * 840), 0, 0, 0);
  };
  // (vector memory of a wavefront completes in order: with the younger item's requests alone under way the older item is there)
  auto arrived = [&]() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DMAS) : "memory");
  };
  int row = row0, g = 0;                             // of the item requested last
  auto advance = [&]() { if (++g == groups) { g = 0; row += rstride; } };

  // x: eight elements a lane and piece, four pieces of every row requested together, the first ones in front of the weight's first items
  constexpr int XP = M <= 2 ? 4 : 2;
  const int pieces = quads * 128;
  for (int p0 = threadIdx.x; p0 - (int)threadIdx.x < pieces; p0 += XP * NW * 64) {
    uint4v v[M][XP];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int c = 0; c < XP; ++c) v[m][c] = __builtin_amdgcn_raw_buffer_load_b128(rows_buffer(a.x + (int64_t)m * a.ldx, a.K * 2), (p0 + c * NW * 64) * 16, 0, 0);
    if (p0 == (int)threadIdx.x) request(0, row, g);
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int c = 0; c < XP; ++c) {
        const int p = p0 + c * NW * 64, e = p * 8;
        const int dst = (m * quads + (e >> 10)) * 1024 + ((e >> 5) & 3) * 256 + ((e >> 7) & 7) * 32 + (e & 31);
        const uint4v r = v[m][c];
        // (elements 0 2 1 3 of every four)
        if (p < pieces)
          *(uint4v*)((_Float16*)smem + dst) = uint4v{__builtin_amdgcn_perm(r[1], r[0], 0x05040100u), __builtin_amdgcn_perm(r[1], r[0], 0x07060302u),
                                                     __builtin_amdgcn_perm(r[3], r[2], 0x05040100u), __builtin_amdgcn_perm(r[3], r[2], 0x07060302u)};
      }
  }
  // (x alone is shared: the first item stays under way)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  float acc[M];
#pragma unroll
  for (int m = 0; m < M; ++m) acc[m] = 0.0f;
  uint32_t low4 = 0x0F0F0F0Fu, low6 = 0x003F003Fu, k1024 = 0x64006400u;
  asm("" : "+v"(low4), "+v"(low6), "+v"(k1024));
  auto work = [&](int at, int wrow, int wg) {
    const char* patch = patches + at * Q6K_PATCH;
    const uint32_t shift = (uint32_t)row_at(wrow) & 3, first = shift + blk * 210;      // of this lane's block of a quad, in bytes
    const char *dwords = patch + (first & ~3u) + 64 * half + 4 * i, *highs = patch + (first & ~3u) + 128 + 32 * half + 4 * i;
    const char *scales = patch + first + 192 + 8 * half + (i >> 2), *ds = patch + first + 208;
    auto dword = [&](const char* p) {
      const uint2v v = *(const q6k_u64*)p;
      return __builtin_amdgcn_alignbyte(v.y, v.x, first);    // (its low two bits)
    };
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int quad = wg * U + u;
      if (quad >= quads) break;
      const uint32_t l0 = dword(dwords + 840 * u), l1 = dword(dwords + 840 * u + 32), h = dword(highs + 840 * u);
      const uint32_t dbits = *(const uint16_t*)(ds + 840 * u);
      float part[M];
#pragma unroll
      for (int m = 0; m < M; ++m) part[m] = 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // codes 32 j + 4 i .. + 3 of the half: low bits from dword j & 1, nibble j >> 1; high bits 2 j, 2 j + 1.  The masks lie in
        // vector registers: an operation with a scalar one takes twice the issue time.
        const uint32_t l = (j & 1 ? l1 : l0) >> (4 * (j >> 1)), hj = j < 2 ? h << (4 - 2 * j) : h >> (2 * j - 4);
        const uint32_t code = __builtin_amdgcn_bitop3_b32(l, hj, low4, 0xE4);          // low4 ? l : hj; bits 6, 7 of a byte are anything
        const half2v off = {(_Float16)1056.0f, (_Float16)1056.0f};                     // 1024 + 32
        const half2v c0 = u2h(__builtin_amdgcn_bitop3_b32(code, low6, k1024, 0xEA)) - off;          // codes 0, 2
        const half2v c1 = u2h(__builtin_amdgcn_bitop3_b32(code >> 8, low6, k1024, 0xEA)) - off;     // codes 1, 3
        int si = *(const int8_t*)(scales + 840 * u + 2 * j);
        asm("" : "+v"(si));                          // (a signed byte load)
        const float s = (float)si;
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const half4 xv = *(const half4*)((const _Float16*)smem + (m * quads + quad) * 1024 + j * 256 + lane * 4);
          float dot = __builtin_amdgcn_fdot2(c0, half2v{xv[0], xv[1]}, 0.0f, false);
          dot = __builtin_amdgcn_fdot2(c1, half2v{xv[2], xv[3]}, dot, false);
          part[m] = fmaf(s, dot, part[m]);
        }
      }
      const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(dbits & (quad * 4 + blk < nblk ? 0xFFFFu : 0)));
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = fmaf(d, part[m], acc[m]);
    }
  };
  auto emit = [&](int wrow) {
    float y = 0.0f;                                  // lane m: row m's sum over the lanes
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
  for (int it = 0; it < items; ++it) {
    const int wrow = row, wg = g;
    advance();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (the reads of the patch that is written next)
    request((it + 1) & 1, row, g);
    arrived();
    work(it & 1, wrow, wg);
    if (wg == groups - 1) emit(wrow);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the last look-ahead writes LDS)
}

static size_t q6k_x(int M, int K) { return (size_t)M * ((K / 256 + 3) / 4) * 2048; }

// Time against the tile kernel's best tiling, us: 1 / 2 / 3 / 4 rows, 4096 x 11008 12.0 / 14.4 / 16.2 / (its x is too large)
// against 24.8 - 25.1 (before: 16.6 / 18.1 / 21.5); 12288 x 4096 13.2 / - / - / 20.8 against 27.2 - 28.0 (17.7, four rows 24.5);
// 32000 x 4096 29.0 against 58 - 60 (36.4); 2048 x 2048 3.9 against 12.6 (5.3).  Four rows are the limit, and 80 KiB of x.
bool gemv_q6k_takes(const RowsArgs& a) {
  return a.M <= 4 && a.gamma == nullptr && a.splitk <= 1 && q6k_x(a.M, a.K) <= 80 * 1024;
}

template <int M, int NW>
static int launch_as(const RowsArgs& a, hipStream_t st, int per_cu, size_t lds) {
  const auto kernel = gemv_q6k_kernel<M, NW, NW == 16 ? 4 : M <= 2 ? 8 : 6>;
  if (!gemv_allow_lds((const void*)kernel, 160 * 1024)) return -101;
  const int need = (a.N + NW - 1) / NW, most = per_cu * gemv_cu_count();
  hipLaunchKernelGGL(kernel, dim3(need < most ? need : most), dim3(NW * 64), lds, st, a);
  return HIP_CHECK_LAUNCH();
}
// As many workgroups of eight wavefronts as a CU's LDS and registers hold (32000 x 4096, one row: 2 / 3 / 4 of them 29.8 / 30.8 /
// 28.6 us); where only one fits, sixteen wavefronts share its x (4096 x 11008, three rows: 17.6 -> 16.2 us), unless eight a CU have
// a row each: sixteen would stand on half of the CUs (300 x 8192, four rows: 8.9 us, with sixteen 12.1, before 10.4).
template <int M>
static int launch(const RowsArgs& a, hipStream_t st) {
  const size_t x = q6k_x(M, a.K), lds = x + 8 * 2 * Q6K_PATCH;
  const int fit = (int)(160 * 1024 / lds), most = M <= 2 ? 4 : 3, per_cu = fit < most ? fit : most;
  return per_cu == 1 && a.N > 8 * gemv_cu_count() ? launch_as<M, 16>(a, st, 1, x + 16 * 2 * Q6K_PATCH) : launch_as<M, 8>(a, st, per_cu, lds);
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
