// Dense projections of the decoder's attention: out = x W (+ resid), 16-bit types, fp32
// accumulation, one rounding.  They stand around the prefill attention (the fused Q/K/V
// projection and W_O with the residual; reference: src/model/mha.py:245-287), whose
// contraction is short (d_model, at most 576) and whose row count is long.
//
// What bounds it: at K = 576 a tile's operands are used for few MFMAs, so a kernel that
// stages both operands per k-step waits on its copies (the library's 256 x 256 kernels ran
// these two shapes at 566 and 410 TFLOP/s).  Here a workgroup of 12 waves keeps its rows of
// x (32 to 128, linear_launch) whole in LDS (128: 147 KB; one workgroup per CU; 256 of them at
// the prefill's 32,768 rows) and has no barrier after they land.  Each wave owns 16 NB columns of a pass of 576 (NB <= 3)
// and all rows: a weight fragment, loaded from L2 two k-steps ahead, feeds 8 MFMAs, so per
// k-step a CU reads 36 KB of weights and 96 KB of LDS under 1,152 cycles of MFMAs per SIMD.
//
// The weights come in MFMA fragment order [N / 16][K / 32][64 lanes][8]: lane 16 q + n holds
// column n, k elements 8 q .. + 7.  The product runs transposed (the weights as the MFMA's A
// operand), so a lane ends with 4 consecutive columns of one row and the rows leave in the
// quad-major order (store_quads48).
#include "../../include/nsmoe.h"
#include "gemm_core.h"
#include "nsmoe_capi_internal.h"

namespace nsmoe {

constexpr int LN_WAVES = 12, LN_THREADS = LN_WAVES * 64;
constexpr int LN_MAX_K = 576;
constexpr int LN_PASS = LN_WAVES * 48;  // columns of a full pass

struct LinearArgs {
  const uint16_t* x;      // [M, K]
  const char* w;          // fragment order
  const uint16_t* resid;  // [M, N] or NULL
  uint16_t* out;          // [M, N]; may be resid itself (each element is read, then written,
                          // by one lane)
  int64_t M;
  int K, N;
};

// 16 MR rows (blockIdx.x), passes blockIdx.y, blockIdx.y + gridDim.y, ...
template <int DT, int MR>
__global__ void __launch_bounds__(LN_THREADS, 3) linear_kernel(LinearArgs a) {
  using M = Mma<DT>;
  using Frag = typename M::Frag;
  __shared__ __attribute__((aligned(1024))) char s_x[MR * 16 * LN_MAX_K * 2];
  const int tid = threadIdx.x, lane = tid & 63, lc = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = a.K, N = a.N, nks = K >> 5;
  const int64_t row0 = (int64_t)blockIdx.x * (16 * MR);
  const int rows = (int)min<int64_t>(16 * MR, a.M - row0);
  const char* zero = (const char*)g_zero_kib + lane * 16;

  // The rows, one contiguous block of x, by 1 KiB LDS-DMA copies.  Slot p of row r holds the
  // row's 16-byte chunk x_slot(p, r): whole groups of 8 chunks XORed with r % 8, so the 16
  // rows a fragment read touches at one chunk fall on distinct bank groups.
  const int cpr = K >> 3, cpr8 = cpr & ~7;
  auto x_slot = [&](int c, int r) { return c < cpr8 ? c ^ (r & 7) : c; };
  {
    const int nslot = 16 * MR * cpr;  // a multiple of 64 (cpr % 4 == 0)
    const uint16_t* src = a.x + row0 * K;
    for (int i = wave; i * 64 < nslot; i += LN_WAVES) {  // uniform
      const int s = i * 64 + lane;
      const int r = s / cpr, p = s - r * cpr;
      async_copy16(r < rows ? (const void*)(src + (int64_t)r * K + x_slot(p, r) * 8)
                            : (const void*)zero,
                   s_x + i * 1024);
    }
  }
  wait_vmcnt<0>();
  __syncthreads();

  const int nblk = N >> 4;
  const char* xl = s_x + lc * cpr * 16;  // this lane's row of row block 0
  const int xstep = 16 * cpr * 16;       // bytes between row blocks (16 rows keep r % 8)
  auto pass = [&](int col0, auto nb_tag) __attribute__((always_inline)) {
    constexpr int NB = decltype(nb_tag)::value;
    const int c0 = col0 + wave * 16 * NB;  // the wave's columns of the pass
    if (c0 >= N) return;
    const int b0 = c0 >> 4;
    struct WSet {
      Frag f[NB];
    };
    auto load_w = [&](int ks) __attribute__((always_inline)) -> WSet {
      WSet w;
#pragma unroll
      for (int j = 0; j < NB; ++j)
        w.f[j] = M::load(b0 + j < nblk ? a.w + ((int64_t)(b0 + j) * nks + ks) * 1024 + lane * 16
                                       : zero);
      return w;
    };
    f32x4 acc[MR][NB];
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto step = [&](int ks, const WSet& w) __attribute__((always_inline)) {
      const char* xs = xl + (x_slot(4 * ks + lg, lc) << 4);
#pragma unroll
      for (int i = 0; i < MR; ++i) {
        const Frag xf = M::load(xs + i * xstep);
#pragma unroll
        for (int j = 0; j < NB; ++j) M::run(acc[i][j], w.f[j], xf);
      }
    };
    WSet w0 = load_w(0), w1 = load_w(min(1, nks - 1));
    for (int ks = 0; ks < nks; ks += 2) {
      step(ks, w0);
      w0 = load_w(min(ks + 2, nks - 1));
      if (ks + 1 < nks) {
        step(ks + 1, w1);
        w1 = load_w(min(ks + 3, nks - 1));
      }
    }
    uint16_t* O = a.out + row0 * N;
    const uint16_t* R = a.resid ? a.resid + row0 * N : nullptr;
    // Whole 16-column blocks: NB of them, or what is left of N.
    const int nb = min(NB, nblk - b0);
#pragma unroll
    for (int i = 0; i < MR; ++i) {
      if (16 * i >= rows) break;  // uniform
      uint32_t lo[3] = {0u, 0u, 0u}, hi[3] = {0u, 0u, 0u};
      const int mq = 16 * i + (lane >> 2);  // this lane's row in the quad order
      const bool in = mq < rows;
      if (NB >= 2 && nb >= 2) {
        if (R) {
          load_quads48(lo, hi, in ? (const char*)(R + (int64_t)mq * N + c0) : nullptr, lane, nb == 3);
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            acc[i][j][0] += unpack2<DT>(lo[j], 0);
            acc[i][j][1] += unpack2<DT>(lo[j], 1);
            acc[i][j][2] += unpack2<DT>(hi[j], 0);
            acc[i][j][3] += unpack2<DT>(hi[j], 1);
          }
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          lo[j] = pack2<DT>(acc[i][j][0], acc[i][j][1]);
          hi[j] = pack2<DT>(acc[i][j][2], acc[i][j][3]);
        }
        store_quads48(lo, hi, in ? (char*)(O + (int64_t)mq * N + c0) : nullptr, lane, nb == 3);
      } else {  // one block: 8 bytes a lane
        const int m = 16 * i + lc;
        if (m < rows) {
          f32x4 v = acc[i][0];
          if (R) {
            const uint2 rv = *(const uint2*)(R + (int64_t)m * N + c0 + 4 * lg);
            v[0] += unpack2<DT>(rv.x, 0);
            v[1] += unpack2<DT>(rv.x, 1);
            v[2] += unpack2<DT>(rv.y, 0);
            v[3] += unpack2<DT>(rv.y, 1);
          }
          *(uint2*)(O + (int64_t)m * N + c0 + 4 * lg) =
              make_uint2(pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3]));
        }
      }
    }
  };
  for (int col0 = (int)blockIdx.y * LN_PASS; col0 < N; col0 += (int)gridDim.y * LN_PASS) {
    const int left = N - col0;
    if (left > 2 * 16 * LN_WAVES) pass(col0, std::integral_constant<int, 3>{});
    else if (left > 16 * LN_WAVES) pass(col0, std::integral_constant<int, 2>{});
    else pass(col0, std::integral_constant<int, 1>{});
  }
}

template <int DT>
static int linear_launch(const LinearArgs& a, hipStream_t s) {
  // One workgroup per CU.  32- and 64-row tiles while they fit one round of the chip; past that
  // 80, 96, 112 or 128 rows, by the time of their rounds: a round of 16 mr rows takes about 4 (mr
  // + 1/2) us at N = 576, so 17,000 rows are one round of 80-row tiles rather than one, half
  // empty, of 128-row ones.  A tile's columns are split over a workgroup per pass while those
  // fit too.  Measured per call, N = 960 and N = 576 with the residual in place, against the
  // library's GEMM (us):
  //   rows   256:   8.6 /   9.0 ( 21 /  18)     4096:  10.7 /   9.7 ( 21 /  18)
  //        10006:  18.9 /  14.8 ( 27 /  18)    16384:  24.7 /  19.1 ( 37 /  27)
  //        17000:  25.4 /  20.2 ( 45 /  22)    20000:  27.9 /  22.0 ( 46 /  24)
  //        24000:  31.9 /  25.1 ( 43 /  41)    28000:  35.8 /  28.7 ( 65 /  48)
  //        32768:  41.2 /  34.1 ( 57 /  46)    36000:  50.6 /  39.9 ( 62 /  54)
  //        50000:  66.3 /  52.0 ( 81 /  64)    65536:  81.8 /  66.3 (110 /  65)
  //        98304: 127.9 /  96.2 (149 / 110)   131072: 167.2 / 134.4 (200 / 127)
  //       262144: 329.9 / 297.1 (391 / 256)
  // (With 128-row tiles alone 17000 rows took 31.5 / 26.7, 36000 65.4 / 54.2.  From 60,000 rows
  // on the library is up to 3 % faster at N = 576, from 131,072 more; every sublayer runs both,
  // and the two together are faster here.)  The 128-row form spills 8 VGPRs; no other does.
  const int64_t cus = device_cus();
  int mr = 2;
  if (cdiv(a.M, 64) > cus) {
    auto cost = [&](int r) { return cdiv(cdiv(a.M, 16 * r), cus) * (2 * r + 1); };
    mr = 8;
    for (int r = 7; r >= 5; --r)
      if (cost(r) < cost(mr)) mr = r;
  } else if (cdiv(a.M, 32) > cus) {
    mr = 4;
  }
  const int64_t tiles = cdiv(a.M, 16 * mr), passes = cdiv(a.N, LN_PASS);
  NSMOE_REQUIRE(tiles < INT32_MAX, "linear: too many rows");
  const dim3 grid((unsigned)tiles, tiles * passes <= cus ? (unsigned)passes : 1u);
  KernelTimer timer("linear", s);
  if (mr == 2) linear_kernel<DT, 2><<<grid, LN_THREADS, 0, s>>>(a);
  else if (mr == 4) linear_kernel<DT, 4><<<grid, LN_THREADS, 0, s>>>(a);
  else if (mr == 5) linear_kernel<DT, 5><<<grid, LN_THREADS, 0, s>>>(a);
  else if (mr == 6) linear_kernel<DT, 6><<<grid, LN_THREADS, 0, s>>>(a);
  else if (mr == 7) linear_kernel<DT, 7><<<grid, LN_THREADS, 0, s>>>(a);
  else linear_kernel<DT, 8><<<grid, LN_THREADS, 0, s>>>(a);
  timer.stop();
  return check_launch("linear_kernel");
}

}  // namespace nsmoe

using namespace nsmoe;

extern "C" int nsmoe_linear(int32_t dtype, const void* x, int64_t n_rows, int32_t k, int32_t n,
                            const void* w_packed, const void* resid, void* out, void* stream) {
  NSMOE_REQUIRE(dtype == DT_BF16 || dtype == DT_F16, "linear: 16-bit types only");
  NSMOE_REQUIRE(n_rows >= 0 && n_rows < ((int64_t)1 << 36), "linear: bad row count");
  NSMOE_REQUIRE(k >= 32 && k % 32 == 0 && k <= LN_MAX_K && n >= 16 && n % 16 == 0 && n <= 65536,
                "linear: takes k %% 32 == 0, k <= %d, n %% 16 == 0 (k %d, n %d)", LN_MAX_K, k, n);
  if (n_rows == 0) return NSMOE_OK;
  NSMOE_REQUIRE(x && w_packed && out, "linear: NULL pointer");
  NSMOE_REQUIRE(((uintptr_t)x & 15) == 0 && ((uintptr_t)w_packed & 15) == 0 &&
                    ((uintptr_t)out & 15) == 0 && ((uintptr_t)resid & 15) == 0,
                "linear: misaligned pointer");
  const LinearArgs a{(const uint16_t*)x, (const char*)w_packed, (const uint16_t*)resid,
                     (uint16_t*)out, n_rows, k, n};
  hipStream_t s = (hipStream_t)stream;
  return dtype == DT_BF16 ? linear_launch<DT_BF16>(a, s) : linear_launch<DT_F16>(a, s);
}
