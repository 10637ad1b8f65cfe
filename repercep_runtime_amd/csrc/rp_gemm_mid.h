// Medium tiles of the FP8 GEMM: products whose grid of 256 x 256 tiles leaves
// CUs idle, narrow N, and a K that ends inside a 64-byte MFMA depth.
// Included by rp_gemm.hip, whose helpers (GemmArgs, the direct-to-LDS load,
// the MFMA and epilogue functions) it uses.
//
// gemm_mid_kernel<BM, KN, EPI, LEAD>: block tiles of BM x 128 (BM 128 or 64) on
// v_mfma_f32_32x32x64_f8f6f4, four waves (2 x 2) of BM/2 x 64 each, C^T tiles
// as in gemm256_kernel (A operand = rows of B^T).  Operands stream by
// direct-to-LDS loads in K slices of 128 bytes through gemm256_kernel's ring
// -- slice kk's A part in slot 2kk mod 5 and its B^T part in slot 2kk + 1
// mod 5, each slice loaded two slices ahead of its use (mod 9 and four ahead
// where a workgroup has its CU to itself, see LEAD) -- but a slot is 16 KiB,
// so two workgroups share a CU and one's waits, fill and stores
// overlap the other's MFMAs.
//
// What bounds it: a wave part of 64 x 64 reads (64 + 64) x 64 operand bytes
// from LDS per four MFMAs (256 cycles), 128 bytes per CU cycle with four
// waves -- the LDS's whole read rate, so these tiles do not reach the
// 256 x 256 kernel's MFMA rate (0.465 us per 128 x 128 x 128 step and CU
// against 1.45 us per 256 x 256 x 128 step).  They win where that kernel's
// tiles are too few or its last round too empty.  Measured, (N, K) B, us:
//     M      N     K    256 x 256   here        M      N      K   256 x 256  here
//    16   5120  5120      46.1       9.6      1024   5120   5120    52.3     33.9
//   128   5120 13824     108.1      22.4      3600   5120   5120   110.1     93.9
//   512   5120  5120      47.4      23.2      3600   8960   1536    69.2     54.1
// and, row-scaled and batched (40 heads), 3600 x 3600 x 128: 406 -> 357;
// 3600 x 128 x 3600: 231 (the VGPR-staged kernel) -> 153.  A 128 x 64 tile
// was slower at N = 64 too (137 against 134), and a two-slot form for K of
// one slice, for more workgroups per CU, slower at 3600 x 3600 x 128 (594).
//
// K may be any multiple of 16: loads past K re-read the last granule (or K
// row) inside it, and the last sub-slice's operands are zeroed past K in
// registers (a re-read byte may be a NaN code, so both operands are).
//
// Split K (kEpiPart): blockIdx.z runs one part of the K slices and writes
// fp32 partial sums to g.part; gemm_reduce_kernel adds the parts in order and
// applies the epilogue.  For small M: a weight-streaming grid of a few dozen
// tiles cannot draw the HBM rate from a few dozen CUs.

constexpr int kEpiPart = 3;   // fp32 partial sums of one K part (no scale)

constexpr int kGmBN = 128;    // columns per tile

// Slices loaded ahead of their use (LEAD): two in the five-slot ring, which
// leaves LDS for a second workgroup on the CU.  A grid of at most a workgroup
// per CU has that LDS to itself: nine slots, four slices ahead, for its loads
// bound it (0.8 us per slice at two ahead when the operands come from HBM).
// us per call, 2 / 4 ahead, weights changing from call to call, (N, K) and
// (K, N) B: 256 x 5120 x 5120 32.3 / 23.8 and 40.1 / 30.1; 512 rows 33.9 /
// 30.3 and 39.8 / 34.7; 256 x 4096 x 4096 25.9 / 17.6 and 26.6 / 21.4; 256 x
// 3072 x 3072 13.9 / 11.0 and 14.6 / 12.6.  The same weights again and again:
// 256 x 5120 x 5120 21.4 / 16.4, but 256 x 4096 x 4096, which the L2s hold,
// 11.3 / 11.7.  Workgroups of few slices lose by the longer fill (16 x 4096 x
// 4096, K parts of 4 slices, 9.1 / 9.7; 512 x 1536 x 8960, of 14, 20.0 /
// 20.7).
constexpr int kGmDeep = 4;
constexpr int kGmDeepSlices = 20;
constexpr int64_t kGmDeepGrid = 256;

template <int BM>
struct GmGeo {
  static constexpr int BN = kGmBN;
  static constexpr int WM = BM / 2, WN = BN / 2;      // a wave's part
  static constexpr int NBM = WM / 32, NBN = WN / 32;  // 32-row operand blocks
  static constexpr int A_HALF = BM * kG2Pitch, B_HALF = BN * kG2Pitch;
  static constexpr int SLOT = A_HALF > B_HALF ? A_HALF : B_HALF;
  static constexpr int ALOADS = A_HALF / 4096, BLOADS = B_HALF / 4096;  // 1 KiB loads per wave
  static constexpr int LOADS = ALOADS + BLOADS;
  // a (K, N) B slice: eight granules (16 N bytes) per 128-byte K row.  Two
  // rows share a sweep of the LDS banks; the granules of row r move by
  // 2 ((r / 2) mod 4), so that eight K rows times two neighbouring granules --
  // one transpose read -- cover the bank groups once
  static constexpr int GRAN = BN / 16;
  static __device__ __forceinline__ int kn_swz(int row) { return 2 * ((row >> 1) & 3); }
  static_assert(BM == 64 || BM == 128, "tile");
};

__device__ __forceinline__ i32x8 gm_kn_operand(uint32_t base) {
  const i32x2 r0 = lds_tr8(base), r1 = lds_tr8(base + 8 * kGmBN);
  const i32x2 r2 = lds_tr8(base + 16 * kGmBN), r3 = lds_tr8(base + 24 * kGmBN);
  return i32x8{r0.x, r0.y, r1.x, r1.y, r2.x, r2.y, r3.x, r3.y};
}

template <int NBM, int NBN>
struct GmOps {
  i32x8 a[NBM], b[NBN];
};

// s_waitcnt vmcnt(max(n, 0)), n at most LOADS * MAX and a multiple of LOADS
template <int LOADS, int MAX>
__device__ __forceinline__ void gm_wait_slices(int left) {
  if (MAX > 0 && left >= MAX) g2_wait_vmem<LOADS * MAX>();
  else if constexpr (MAX > 0) gm_wait_slices<LOADS, MAX - 1>(left);
  else g2_wait_vmem<0>();
}

template <int BM, bool KN, int EPI, int LEAD>
__global__ __launch_bounds__(kG2Threads) __attribute__((amdgpu_waves_per_eu(LEAD > 2 ? 1 : 2, 2)))
void gemm_mid_kernel(GemmArgs g) {
  using G = GmGeo<BM>;
  constexpr int BN = kGmBN, SLOTS = 2 * LEAD + 1, NBM = G::NBM, NBN = G::NBN, SLOT = G::SLOT;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[SLOTS * SLOT];
  const uint32_t smem_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem;

  gemm_batch(g);
  // XCD-aware remap, then a column-major walk over bands of C of g.band tiles
  const int nwork = g.tiles_m * g.tiles_n;
  const int w = blockIdx.x;
  const int per = nwork >> 3, rem = nwork & 7;
  const int xcd = w & 7;
  const int L = xcd * per + min(xcd, rem) + (w >> 3);
  const int band_tiles = g.band * g.tiles_n;
  const int band = L / band_tiles;
  const int in_band = L - band * band_tiles;
  const int band_h = min(g.band, g.tiles_m - band * g.band);
  const int tm = band * g.band + in_band % band_h;
  const int tn = in_band / band_h;
  const int64_t m0 = (int64_t)tm * BM;
  const int64_t n0 = (int64_t)tn * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane & 31, lg = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;

  // this workgroup's K slices [s0, s0 + nslice) (all of them but for kEpiPart)
  const int s0 = EPI == kEpiPart ? (int)blockIdx.z * g.part_slices : 0;
  const int64_t k_left = g.K - (int64_t)s0 * kG2K;
  const int64_t k_own = EPI == kEpiPart ? min(k_left, (int64_t)g.part_slices * kG2K) : k_left;

  // This lane's loads, as in gemm256_kernel: A and (N, K) B^T eight lanes per
  // row's 128-byte slice, K granule slot ^ ((r >> 1) & 7) of row r at `slot`;
  // (K, N) B GRAN lanes per K row, N granule slot ^ kn_swz(r) at `slot`.
  // Rows past M or N re-read the last row, N granules past N the last one.
  const uint8_t* abase = g.a + m0 * g.lda + (int64_t)s0 * kG2K;
  const uint8_t* bbase = KN ? g.bt + n0 + (int64_t)s0 * kG2K * g.ldb
                            : g.bt + n0 * g.ldb + (int64_t)s0 * kG2K;
  uint32_t gofs[G::LOADS];
#pragma unroll
  for (int n = 0; n < G::LOADS; ++n) {
    const bool is_a = n < G::ALOADS;
    const int p = ((is_a ? n : n - G::ALOADS) * 4 + wave) * kWave + lane;
    if (KN && !is_a) {
      const int row = p / G::GRAN, slot = p % G::GRAN;
      const int last = (int)min((g.N - n0) >> 4, (int64_t)G::GRAN) - 1;
      gofs[n] = (uint32_t)(row * g.ldb + min(slot ^ G::kn_swz(row), last) * 16);
      continue;
    }
    const int row = p >> 3, slot = p & 7;
    const int s16 = (slot ^ ((row >> 1) & 7)) * 16;
    gofs[n] = is_a ? (uint32_t)((min(m0 + row, g.M - 1) - m0) * g.lda + s16)
                   : (uint32_t)((min(n0 + row, g.N - 1) - n0) * g.ldb + s16);
  }
  const int nsub = (int)((k_own + kG2Sub - 1) / kG2Sub);
  const int nslice = (nsub + 1) >> 1;
  const int ktail = (int)(k_own - (int64_t)(nsub - 1) * kG2Sub);     // K of the last sub-slice
  const int krows = (int)(k_own - (int64_t)(nslice - 1) * kG2K);     // and of the last slice
  // what an A or (N, K) load of the last slice steps back to stay inside K:
  // this lane's K granule is the same in all of them (the block's parity,
  // bit 2 of the swizzle, is the wave's)
  const int kg = (lane & 7) ^ (((wave & 1) << 2) | ((lane >> 4) & 3));
  const uint32_t back = (uint32_t)max(kg - (krows / 16 - 1), 0) * 16;
  // load n of slice kk into `slot`
  auto issue = [&](int n, int kk, int slot, auto full_c) __attribute__((always_inline)) {
    constexpr bool FULL = decltype(full_c)::value;
    const bool is_a = n < G::ALOADS;
    const int b = is_a ? n : n - G::ALOADS;
    uint32_t off = gofs[n];
    if (!FULL && kk == nslice - 1) {
      if (KN && !is_a) {
        const int row = ((b * 4 + wave) * kWave + lane) / G::GRAN;
        off -= (uint32_t)(max(row - (krows - 1), 0) * g.ldb);
      } else {
        off -= back;
      }
    }
    const uint8_t* src = is_a ? abase + (int64_t)kk * kG2K
                              : bbase + (int64_t)kk * kG2K * (KN ? g.ldb : 1);
    g2_gload_lds16_s(src, off, smem_lds + (uint32_t)(slot * SLOT + (b * 4 + wave) * 1024));
  };

  // per-lane operand offsets inside a slot (see gemm256_kernel)
  const int swz = (lq >> 1) & 7;
  const int h00 = ((2 * lg) ^ swz) * 16, h01 = ((2 * lg + 1) ^ swz) * 16;
  const int h10 = ((4 + 2 * lg) ^ swz) * 16, h11 = ((4 + 2 * lg + 1) ^ swz) * 16;
  const int a_off = (wm * G::WM + lq) * kG2Pitch;
  const int b_off = (wn * G::WN + lq) * kG2Pitch;
  uint32_t kn_off[NBN];
  {
    const int i = lane & 15;
    const int row = 32 * lg + (i >> 1);
#pragma unroll
    for (int j = 0; j < NBN; ++j) {
      const int gr = 2 * NBN * wn + 2 * j + ((lane >> 4) & 1);
      // kn_swz(row): the rows of one read differ in i >> 1 alone
      kn_off[j] = (uint32_t)(row * BN + ((gr ^ G::kn_swz(i >> 1)) << 4) + 8 * (i & 1));
    }
  }
  auto b_op = [&](const uint8_t* st, int j, int h, int c0, int c1) __attribute__((always_inline)) {
    if constexpr (KN) {
      const uint32_t st_lds = smem_lds + (uint32_t)(st - smem);
      return gm_kn_operand(st_lds + kn_off[j] + (uint32_t)(64 * h * BN));
    } else {
      return g2_op(st + b_off + 32 * j * kG2Pitch, c0, c1);
    }
  };
  auto wrap = [](int x) { return x >= SLOTS ? x - SLOTS : x; };

  f32x16 acc[NBM][NBN];
#pragma unroll
  for (int i = 0; i < NBM; ++i)
#pragma unroll
    for (int j = 0; j < NBN; ++j) acc[i][j] = f32x16{};

#pragma unroll
  for (int s = 0; s < LEAD; ++s)
    if (s < nslice) {
#pragma unroll
      for (int n = 0; n < G::LOADS; ++n)
        issue(n, s, 2 * s + (n < G::ALOADS ? 0 : 1), std::false_type{});
    }
  gm_wait_slices<G::LOADS, LEAD - 1>(nslice - 1);   // slice 0 has landed
  __syncthreads();
  GmOps<NBM, NBN> o0, o1;
#pragma unroll
  for (int i = 0; i < NBM; ++i) o0.a[i] = g2_op(smem + a_off + 32 * i * kG2Pitch, h00, h01);
#pragma unroll
  for (int j = 0; j < NBN; ++j) o0.b[j] = b_op(smem + SLOT, j, 0, h00, h01);

  auto zero_tail = [&](GmOps<NBM, NBN>& o) __attribute__((always_inline)) {
    const bool lo = 32 * lg < ktail, hi = 32 * lg + 16 < ktail;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int i = 0; i < NBM; ++i) o.a[i][e] = (e < 4 ? lo : hi) ? o.a[i][e] : 0;
#pragma unroll
      for (int j = 0; j < NBN; ++j) o.b[j][e] = (e < 4 ? lo : hi) ? o.b[j][e] : 0;
    }
  };

  // Sub-step (kk, H), gemm256_kernel's schedule: the MFMAs of sub-slice
  // 2kk + H on `cur`, the operand reads of the next sub-slice into `nxt`
  // (in the first half of the MFMAs) and the loads of slice kk + LEAD's A part
  // (H = 0) or B^T part (H = 1).  (kk, 1) begins with the slice's one wait and
  // barrier: slice kk + 1 has landed, and every wave has read slice kk.
  int sa = 0;   // slot of slice kk's A part
  auto sub = [&](int kk, auto Hc, auto Sc, GmOps<NBM, NBN>& cur, GmOps<NBM, NBN>& nxt)
      __attribute__((always_inline)) {
    constexpr int H = decltype(Hc)::value;
    constexpr bool STEADY = decltype(Sc)::value;
    const int u = 2 * kk + H;
    const bool more = STEADY || u + 1 < nsub;
    const bool load = STEADY || kk + LEAD < nslice;
    if (!STEADY && !more && ktail < kG2Sub) zero_tail(cur);
    if (H == 1) {
      if (more) {
        // slices kk + 2 and on may stay in flight
        if (load) g2_wait_vmem<(LEAD - 2) * G::LOADS + G::ALOADS>();
        else gm_wait_slices<G::LOADS, LEAD - 2>(nslice - 2 - kk);
      }
      __syncthreads();
    }
    const uint8_t* sta = smem + (H == 0 ? sa : wrap(sa + 2)) * SLOT;
    const uint8_t* stb = smem + (H == 0 ? wrap(sa + 1) : wrap(sa + 3)) * SLOT;
    const int lslot = H == 0 ? wrap(sa + 2 * LEAD) : sa;
    const int r0 = H == 0 ? h10 : h00, r1 = H == 0 ? h11 : h01;
    constexpr int NM = NBM * NBN;                        // MFMAs of the sub-step
    constexpr int NL = H == 0 ? G::ALOADS : G::BLOADS;   // loads
    constexpr int NR = NBM + NBN;                        // operand reads
    constexpr int RM = NM > 1 ? NM / 2 : 1;              // MFMAs they spread over
#pragma unroll
    for (int t = 0; t < NM; ++t) {
      const int i = t / NBN, j = t % NBN;
      acc[i][j] = mfma_32x32x64(cur.b[j], cur.a[i], acc[i][j]);
      if (t < RM && more) {
#pragma unroll
        for (int x = t * NR / RM; x < (t + 1) * NR / RM; ++x) {
          if (x < NBM) nxt.a[x] = g2_op(sta + a_off + 32 * x * kG2Pitch, r0, r1);
          else nxt.b[x - NBM] = b_op(stb, x - NBM, H == 0 ? 1 : 0, r0, r1);
        }
      }
      if (load) {
#pragma unroll
        for (int x = t * NL / NM; x < (t + 1) * NL / NM; ++x)
          issue((H == 0 ? 0 : G::ALOADS) + x, kk + LEAD, lslot,
                std::integral_constant<bool, STEADY>{});
      }
      if constexpr (STEADY) __builtin_amdgcn_sched_barrier(0);
    }
    if (H == 1) sa = wrap(sa + 2);
  };
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  const int nfull = nsub >> 1;
  int kk = 0;
  const int nsteady = max(0, nslice - 1 - LEAD);
  for (; kk < nsteady; ++kk) {
    sub(kk, H0{}, std::true_type{}, o0, o1);
    sub(kk, H1{}, std::true_type{}, o1, o0);
  }
  for (; kk < nfull; ++kk) {
    sub(kk, H0{}, std::false_type{}, o0, o1);
    sub(kk, H1{}, std::false_type{}, o1, o0);
  }
  if (nsub & 1) sub(nfull, H0{}, std::false_type{}, o0, o1);

  if constexpr (EPI == kEpiPart) {
    float* const part = g.part + (int64_t)blockIdx.z * g.M * g.N;
#pragma unroll
    for (int i = 0; i < NBM; ++i) {
      const int64_t m = m0 + wm * G::WM + 32 * i + lq;
      if (m >= g.M) continue;
#pragma unroll
      for (int j = 0; j < NBN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int64_t n = n0 + wn * G::WN + 32 * j + 8 * q + 4 * lg;
          if (n < g.N)
            *reinterpret_cast<f32x4*>(part + m * g.N + n) =
                f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                      acc[i][j][4 * q + 3]};
        }
    }
    return;
  }

  // epilogue: the bf16 tile through LDS, as in gemm256_kernel.  A row of a
  // wave's part is 64 bf16 = 128 bytes, two rows per sweep of the banks;
  // 8-byte slot s of row r sits at s ^ cswz(r), cswz(r) = (r / 2) mod 16, so a
  // half-wave's 32 rows fill the banks once
  constexpr bool ROWS = EPI == kEpiRows;
  const float scale = ROWS ? 1.0f
                    : (g.a_dev ? *g.a_dev : g.a_scale) * (g.b_dev ? *g.b_dev : g.b_scale);
  constexpr int PITCH = 2 * G::WN;
  static_assert(4 * G::WM * PITCH <= SLOTS * SLOT, "C staging fits the slots");
  uint8_t* const ct = smem + wave * G::WM * PITCH;
  auto cswz = [](int r) { return (r >> 1) & 15; };
  float sm[NBM];
#pragma unroll
  for (int i = 0; i < NBM; ++i) {
    const int64_t m = m0 + wm * G::WM + 32 * i + lq;
    sm[i] = ROWS && m < g.M ? g.row_scale[m] : 1.0f;
  }
  __syncthreads();   // every wave has finished reading the operand slots
#pragma unroll
  for (int j = 0; j < NBN; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t n = n0 + wn * G::WN + 32 * j + 8 * q + 4 * lg;
      if (EPI != kEpiPlain && n >= g.N) continue;   // never stored, nor its scales read
      const uint2 bb = EPI == kEpiBias ? bias4(g, n) : make_uint2(0u, 0u);
      const float4 sn = ROWS ? *reinterpret_cast<const float4*>(g.col_scale + n)
                             : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int i = 0; i < NBM; ++i) {
        const f32x16& v = acc[i][j];
        float o[4];
        if constexpr (ROWS)
          epi4_rows(false, bb, sm[i], sn, v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3], o);
        else
          epi4(EPI == kEpiBias, bb, scale, v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3], o);
        const uint2 pk = make_uint2(g2_pack_bf16(o[0], o[1]), g2_pack_bf16(o[2], o[3]));
        const int r = 32 * i + lq;
        *reinterpret_cast<uint2*>(ct + r * PITCH + ((8 * j + 2 * q + lg) ^ cswz(lq)) * 8) = pk;
      }
    }
  __syncthreads();
  const bool c16 = reinterpret_cast<uintptr_t>(g.c) % 16 == 0 && g.ldc % 8 == 0;
  constexpr int LPR = PITCH / 16;       // lanes per row, 16 bytes each
  constexpr int RPS = kWave / LPR;      // rows per store instruction
  const int c = lane % LPR;
  const int64_t n = n0 + wn * G::WN + 8 * c;
  // logical slots 2c, 2c + 1 of row r: granule c ^ (cswz(r) >> 1), swapped
  // when cswz(r) is odd
  auto stage_row = [&](int r) __attribute__((always_inline)) {
    const int sw = cswz(r & 31);
    const uint4 t = *reinterpret_cast<const uint4*>(ct + r * PITCH + (c ^ (sw >> 1)) * 16);
    return sw & 1 ? u32x4{t.z, t.w, t.x, t.y} : u32x4{t.x, t.y, t.z, t.w};
  };
  if (c16 && m0 + BM <= g.M && n0 + BN <= g.N) {
    uint16_t* const cw = g.c + (m0 + wm * G::WM) * g.ldc + n;
    constexpr int NST = G::WM / RPS, U = NST < 8 ? NST : 8;
#pragma unroll
    for (int k8 = 0; k8 < NST; k8 += U) {
      u32x4 t[U];
#pragma unroll
      for (int u = 0; u < U; ++u) t[u] = stage_row(RPS * (k8 + u) + lane / LPR);
#pragma unroll
      for (int u = 0; u < U; ++u)
        __builtin_nontemporal_store(
            t[u], reinterpret_cast<u32x4*>(cw + (int64_t)(RPS * (k8 + u) + lane / LPR) * g.ldc));
    }
    return;
  }
#pragma unroll 4
  for (int k = 0; k < G::WM / RPS; ++k) {
    const int r = RPS * k + lane / LPR;
    const int64_t m = m0 + wm * G::WM + r;
    const u32x4 t = stage_row(r);
    if (m >= g.M || n >= g.N) continue;
    uint16_t* dst = g.c + m * g.ldc + n;
    if (c16 && n + 8 <= g.N) {
      __builtin_nontemporal_store(t, reinterpret_cast<u32x4*>(dst));
    } else {
      // rows off 16 bytes share their cache lines with the neighbouring tile:
      // kept in L2, the halves of a line leave together (non-temporal / plain,
      // us: 40 x 2500 x 2500 of K = 64 420 / 235, 8 x 2500 x 2500 81 / 39,
      // 20000 x 3076 of K = 512 102 / 60; 40 x 2500 x 2500 of K = 512 loses,
      // 294 / 343, and takes the large tiles, 300)
      *reinterpret_cast<u32x2*>(dst) = u32x2{t.x, t.y};
      if (n + 8 <= g.N)   // N % 4 == 0
        *reinterpret_cast<u32x2*>(dst + 4) = u32x2{t.z, t.w};
    }
  }
}

// C = bf16(epilogue(sum of the K parts, in order)): one thread per four
// columns of a row.
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmArgs g, int parts) {
  const int64_t n4 = g.N >> 2;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= g.M * n4) return;
  const int64_t m = t / n4, n = (t - m * n4) * 4;
  const float* p = g.part + m * g.N + n;
  f32x4 v = *reinterpret_cast<const f32x4*>(p);
  for (int s = 1; s < parts; ++s)
    v += *reinterpret_cast<const f32x4*>(p + (int64_t)s * g.M * g.N);
  const float scale = (g.a_dev ? *g.a_dev : g.a_scale) * (g.b_dev ? *g.b_dev : g.b_scale);
  float o[4];
  epi4(g.bias != nullptr, g.bias ? bias4(g, n) : make_uint2(0u, 0u), scale, v[0], v[1], v[2],
       v[3], o);
  *reinterpret_cast<uint2*>(g.c + m * g.ldc + n) =
      make_uint2(g2_pack_bf16(o[0], o[1]), g2_pack_bf16(o[2], o[3]));
}
