// Row-wise scaled FP8 GEMM for few output tiles (short token counts): one tile per workgroup,
// K stages in a deep LDS ring.  Same operands, products and epilogue as
// gemm_fp8_rowwise_kernel (gemm.hip), and the same bits: every output sums the same products
// in the same order.
//
// What bounds such a product is not bandwidth or matrix-core rate but the chain of K stages:
// with fewer tiles than CUs a workgroup is alone on its CU, and with two stage buffers each
// stage waits out one copy's latency (1.07 us per 128 bytes of K on MI355X, weights from
// HBM).  Here the tile is small enough to give every CU one, the ring keeps NS - 1 stages of
// copies in flight, and a stage's fragments are read from LDS while the previous stage's
// products run, so a stage costs 0.25-0.55 us (by tile size, gemm_pick).  MI355X, weights
// from HBM, before -> after: 1 x 3072 x 3072 16.7 -> 8.0 us, 512 x 3072 x 3072 18.9 -> 11.7,
// 1 x 9216 x 3072 23.2 -> 10.3, 256 x 9216 x 3072 26.6 -> 19.9, 1 x 3072 x 12288 83.6 -> 23.6,
// 1024 x 3072 x 12288 103.7 -> 64.7 us.  Splitting K over workgroups would shorten the chain
// further, but would sum the products in another order.
#pragma once

namespace mxf8 {

// Block tile BM (tokens) x BN (channels) on WM x WN waves of (BM / WM) x (BN / WN); NS stages
// of 128 U bytes of K in the ring (U = 2 halves the barriers where a stage has few products).
template <int BM_, int BN_, int WM_, int WN_, int NS_, int U_>
struct GemmRing {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, NS = NS_, U = U_;
  static constexpr int NW = WM * WN;
  static constexpr int THREADS = 64 * NW;
  static constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  static constexpr int SUB = (BM + BN) * GEMM_BK;           // LDS bytes per 128 bytes of K (W rows, then X rows)
  static constexpr int STAGE = U * SUB, BK = U * GEMM_BK;
  static constexpr int DMA_PER_WAVE = U * ((BM + BN) / 8 / NW);  // 1 KB DMA instructions per wave per stage
  static constexpr int OUT_PITCH = BN * 2 + 16;             // staged output row bytes
  static constexpr int EP = 2 * BN + BM;                    // epilogue operands (fp32): scales, bias, token scales
  static_assert(NS * STAGE + EP * 4 <= 160 * 1024, "LDS ring");
  static_assert(BM * OUT_PITCH <= NS * STAGE, "output staging");
  static_assert((BM + BN) / 8 % NW == 0 && BN % 16 == 0, "DMA shares");
  static_assert(NS >= 3 && (NS - 1) * DMA_PER_WAVE < 64, "vmcnt counts the copies of NS - 1 stages");

  // This wave's share of one stage, as gemm_dma, but whichever operand each instruction's 8
  // rows belong to.
  static __device__ __forceinline__ void dma(__amdgpu_buffer_rsrc_t wrs, __amdgpu_buffer_rsrc_t xrs, uint8_t* stage,
                                             const uint32_t (&lane_off)[2], int K, int wave, int k0) {
    constexpr int PER_SUB = DMA_PER_WAVE / U;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < PER_SUB; ++j) {
        const int J = wave * PER_SUB + j;
        const bool is_w = J < BN / 8;
        const __amdgpu_buffer_rsrc_t rs = is_w ? wrs : xrs;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, LDS_PTR(stage + u * SUB + J * 1024), 16, lane_off[J & 1],
                                                 (is_w ? 8 * J : 8 * J - BN) * K + k0 + u * GEMM_BK, 0, 0);
      }
  }
};

template <class C, int ACT, bool LORA, bool KTAIL>
__global__ __launch_bounds__(C::THREADS) void gemm_ring_kernel(
    const uint8_t* __restrict__ a8, const uint8_t* __restrict__ w8, const float* __restrict__ sa,
    const float* __restrict__ sw, const uint16_t* __restrict__ bias, const uint16_t* __restrict__ lora_t,
    const uint16_t* __restrict__ lora_b, int lora_r, float lora_scale, uint16_t* __restrict__ out, int M, int N,
    int K, int64_t ld_out, int tiles_m, int tiles_n, int group_m) {
  constexpr int TM = C::TM, TN = C::TN, NS = C::NS;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NS * C::STAGE];
  __shared__ __attribute__((aligned(16))) float ep[C::EP];  // channel scales [BN], bias [BN], token scales [BM]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wn = wave / C::WM, wm = wave % C::WM;
  const int wrow0 = wn * (C::BN / C::WN), xrow0 = wm * (C::BM / C::WM);
  const int nk = (K + C::BK - 1) / C::BK;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, group_m, tm, tn);
  const int m0 = tm * C::BM, n0 = tn * C::BN;
  uint32_t lane_off[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    lane_off[par] = (uint32_t)((lane >> 3) * K) +
                    (uint32_t)(((lane & 7) ^ lds_swz<GEMM_BK>(8 * par + (lane >> 3))) << 4);
  auto rsrc = [&](const uint8_t* base, int row0, int rows, int span) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)(base + (int64_t)row0 * K), 0, min(rows - row0, span) * K,
                                             0x00020000);
  };
  const __amdgpu_buffer_rsrc_t wrs = rsrc(w8, n0, N, C::BN), xrs = rsrc(a8, m0, M, C::BM);
  // The epilogue's operands are read first and handed over through LDS while the first
  // stages are in flight (indices past M or N read the last element; those outputs are not
  // stored).
  // (Unconditional loads from selected addresses: a load under a condition would be waited
  // for where the condition ends, before the first copy is issued.)
  constexpr int NEP = (C::EP + C::THREADS - 1) / C::THREADS;
  float epv[NEP];
  uint16_t epb[NEP];
#pragma unroll
  for (int e = 0; e < NEP; ++e) {
    const int i = min((int)threadIdx.x + e * C::THREADS, C::EP - 1);
    const int ch = min(n0 + (i < C::BN ? i : i < 2 * C::BN ? i - C::BN : 0), N - 1);
    epv[e] = *(i < 2 * C::BN ? sw + ch : sa + min(m0 + i - 2 * C::BN, M - 1));
    epb[e] = *(bias ? bias + ch : reinterpret_cast<const uint16_t*>(sw));
  }
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (s < nk) C::dma(wrs, xrs, smem + s * C::STAGE, lane_off, K, wave, s * C::BK);
#pragma unroll
  for (int e = 0; e < NEP; ++e) {
    const int i = threadIdx.x + e * C::THREADS;
    if (i < C::EP)
      ep[i] = i < C::BN || i >= 2 * C::BN ? epv[e] : bias ? bf16_bits_to_f32(epb[e]) : 0.0f;
  }

  v16f acc[TN][TM];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.0f;
  const int r = lane & 31, g = lane >> 5;
  // Fragments of one stage: 64-byte halves h of K.
  struct Frags {
    v8i a[2 * C::U][TN], b[2 * C::U][TM];
  };
  auto read = [&](const uint8_t* st, Frags& f) {
#pragma unroll
    for (int h = 0; h < 2 * C::U; ++h) {
      const uint8_t* sub = st + (h >> 1) * C::SUB;
#pragma unroll
      for (int a = 0; a < TN; ++a) f.a[h][a] = lds_frag(sub, wrow0 + 32 * a + r, 4 * (h & 1) + 2 * g);
#pragma unroll
      for (int b = 0; b < TM; ++b) f.b[h][b] = lds_frag(sub + C::BN * GEMM_BK, xrow0 + 32 * b + r, 4 * (h & 1) + 2 * g);
    }
  };
  // Stage ks's share of this wave's copies has landed once at most the later stages' are in
  // flight (stages up to min(ks + NS - 1, nk - 1) were issued); after the barrier every
  // wave's has, and every wave has read the stage before it.
  auto landed = [&](int ks, auto in_flight) {
    if (ks + decltype(in_flight)::value >= nk)
      wait_vm0();
    else
      wait_vm<decltype(in_flight)::value * C::DMA_PER_WAVE>();
    block_barrier();
    if (KTAIL && ks == nk - 1) {
#pragma unroll
      for (int u = 0; u < C::U; ++u)  // (a part wholly past K is zeroed whole)
        zero_tail<C>(smem + (ks % NS) * C::STAGE + u * C::SUB, (K - ks * C::BK - u * GEMM_BK) >> 4);
      block_barrier();
    }
  };
  auto products = [&](const Frags& f) {
#pragma unroll
    for (int h = 0; h < 2 * C::U; ++h)
#pragma unroll
      for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f.a[h][a], f.b[h][b], acc[a][b], 0, 0, 0, 0, 0, 0);
  };
  int slot = 0;  // ks % NS
  Frags f0, f1;
  landed(0, std::integral_constant<int, NS - 1>{});
  read(smem, f0);
  // One stage: its fragments are in registers (`cur`), so once every wave is here its slot
  // takes stage ks + NS; the next stage's fragments are read while its products run.
  auto stage = [&](int ks, const Frags& cur, Frags& nxt) {
    const int next = slot + 1 == NS ? 0 : slot + 1;
    if (ks + 1 < nk) {
      landed(ks + 1, std::integral_constant<int, NS - 2>{});
      if (ks + NS < nk) C::dma(wrs, xrs, smem + slot * C::STAGE, lane_off, K, wave, (ks + NS) * C::BK);
      read(smem + next * C::STAGE, nxt);
    }
    slot = next;
    products(cur);
  };
  for (int ks = 0; ks < nk; ks += 2) {
    stage(ks, f0, f1);
    if (ks + 1 < nk) stage(ks + 1, f1, f0);
  }

  // ---- epilogue: acc[a][b] register i is channel n0 + wrow0 + 32 a + 8 (i/4) + 4 g + i%4 of
  // token m0 + xrow0 + 32 b + r
  const bool vec = ((N | (int)ld_out) & 7) == 0 && ((uintptr_t)out & 15) == 0;
  block_barrier();  // every wave has read its last fragments: the ring takes the output tile
#pragma unroll
  for (int a = 0; a < TN; ++a) {
#pragma unroll
    for (int b = 0; b < TM; ++b) {
      const float sam = ep[2 * C::BN + xrow0 + 32 * b + r];
      v16f lacc;
      if constexpr (LORA) {
        const uint16_t* brow = lora_b + (int64_t)min(n0 + wrow0 + 32 * a + r, N - 1) * lora_r + 8 * g;
        const uint16_t* trow = lora_t + (int64_t)min(m0 + xrow0 + 32 * b + r, M - 1) * lora_r + 8 * g;
        lora_rows_mma<4>(brow, trow, lora_r, lacc);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int nl = wrow0 + 32 * a + 8 * q + 4 * g;
        *reinterpret_cast<uint2*>(smem + (xrow0 + 32 * b + r) * C::OUT_PITCH + 2 * nl) =
            gemm_out_quad<ACT, LORA>(quad4(acc[a][b], q), q, lacc, sam, *reinterpret_cast<const v4f*>(ep + nl),
                                     *reinterpret_cast<const v4f*>(ep + C::BN + nl), lora_scale);
      }
    }
  }
  block_barrier();
  constexpr int CPR = C::BN / 8;  // 16-byte chunks per staged row
  for (int x = threadIdx.x; x < C::BM * CPR; x += C::THREADS) {
    const int row = x / CPR, c = x % CPR, m = m0 + row, n = n0 + 8 * c;
    if (m >= M || n >= N) continue;
    const uint4 v = *reinterpret_cast<const uint4*>(smem + row * C::OUT_PITCH + 16 * c);
    uint16_t* dst = out + (int64_t)m * ld_out + n;
    if (vec) {
      *reinterpret_cast<uint4*>(dst) = v;
    } else {
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (n + e < N) dst[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
    }
  }
}

// ---- dispatch (gemm_pick chooses) ------------------------------------------------------
// Tiles of the ring kernel, smallest first.
typedef GemmRing<32, 64, 1, 2, 4, 2> GemmRing32x64;     // 96 KB of LDS: one workgroup per CU
typedef GemmRing<64, 64, 2, 2, 4, 1> GemmRing64x64;     // 64 KB: two
typedef GemmRing<128, 64, 4, 2, 3, 1> GemmRing128x64;   // 72 KB: two
typedef GemmRing<128, 128, 2, 4, 4, 1> GemmRing128x128; // 128 KB: one

template <class C>
static void launch_gemm_ring(int act, const uint8_t* a8, const uint8_t* w8, const float* sa,
                             const float* sw, const uint16_t* bias, const uint16_t* lt, const uint16_t* lb, int r,
                             float ls, uint16_t* out, int M, int N, int K, int64_t ld_out, hipStream_t st) {
  const int tiles_m = (int)cdiv(M, C::BM), tiles_n = (int)cdiv(N, C::BN);
  const bool lora = lt != nullptr, ktail = K % C::BK != 0;
#define MXF8_RING_CASE(A, L, T)                                                                                     \
  if (act == A && lora == L && ktail == T) {                                                                        \
    gemm_ring_kernel<C, A, L, T><<<dim3(tiles_m * tiles_n), dim3(C::THREADS), 0, st>>>(                             \
        a8, w8, sa, sw, bias, lt, lb, r, ls, out, M, N, K, ld_out, tiles_m, tiles_n, RING_GROUP_M);                 \
    return;                                                                                                         \
  }
#define MXF8_RING_CASES(A, L) MXF8_RING_CASE(A, L, false) MXF8_RING_CASE(A, L, true)
  MXF8_RING_CASES(MXF8_ACT_NONE, false)
  MXF8_RING_CASES(MXF8_ACT_NONE, true)
  MXF8_RING_CASES(MXF8_ACT_GELU_TANH, false)
  MXF8_RING_CASES(MXF8_ACT_GELU_TANH, true)
#undef MXF8_RING_CASES
#undef MXF8_RING_CASE
}

}  // namespace mxf8
