// Row tiles of 32, 64 or 128 rows over the tile stream (included by mtc_gemm.hip, inside its
// namespace): fp32 results for any M (k_gemm_f32) and bf16 prefill with few rows (k_gemm_tile_short and its
// group and batch kernels).
//
// Block = one TM x 256 output tile over a run of K-steps. Every wave decodes and every
// wave multiplies: a thread takes one cell of a step (512 cells; half a cell where a block has 1024
// threads), whose descriptor was loaded four steps and whose payload three steps ahead (two and one for
// fp32 results in 128 rows), decodes it into the B tile in LDS, and after the barrier the waves run the
// step's MFMAs. With few rows a step's MFMAs take less time than its decode and its memory latency; four
// waves that decode for eight that multiply (k_gemm_tile) then leave most of a CU's issue slots idle. Sums run in k_gemm_tile's order: the same bits for the same K splits.
// Measured against k_gemm_tile's blocks of 64 or 128 rows and their plan, us a call replayed from a graph of ten:
// 2072 x 5472 uniform, M = 40: 23.0 -> 14.9 (20.9 with the old plan's 11 splits; eager, bound by the host, 23.6 ->
// 21.2); 6144 x 1024 QT, M = 160: 27.7 -> 18.9; 4096 x 4096 QT-P, M = 128: 29.0 -> 25.6; 4096 x 4096 QT, M = 256:
// 29.1 -> 29.0 (64 rows, 4 splits: 24.4 us of 16 steps, first data and partials, 5.0 of reduction).
//
// fp32 results on the bf16 matrix cores. A float is cut into bf16 planes by truncation, hi + mid + lo,
// each the upper half of what the planes before left (8 + 8 + 8 significant bits: exact, mid below 2^-7 and
// lo below 2^-15 of hi's leading bit). X takes three planes; a weight code * scale with a code of at most
// 8 bits and a bf16 scale has at most 16 significant bits and takes two, a P16 code or an fp32 scale three.
// Products of bf16 values are exact in fp32, and every pair of planes is multiplied but lo.lo of
// three-plane weights (below 2^-30 of the product). v_mfma_f32_32x32x16_bf16 does 16 times the products
// per clock of v_mfma_f32_16x16x4f32, for six or eight times the number.
//   Two accumulators: hi.hi in one, the other pairs in a second that is added at the end. In one, the small
// pairs of a slice fall below half an ulp of a long sum of one sign, always to the same side.
//   X and the scales are multiplied by 2^24 first and the sums by 2^-48 at the end: then every bit of an
// fp32 value, of a subnormal one too, is a normal bf16 number, where the low planes of values under 2^-109
// would lose bits below 2^-133. X or weights that are not finite have no planes (inf - inf), and values from
// 2^104 or sums from 2^80 on overflow: a block that met one computes its tile again in plain fp32.
// Error against fp64, 2-norm, 4096 x 4096 QT @ 4.5 (an fma chain in K order: the fp32 MFMAs of 16-row tiles):
// M = 100 1.2e-7 (6.0e-7), M = 2048 3.4e-7 (1.0e-6); X and W positive, M = 2048 3.0e-7 (8.6e-7), 8192 x 4096
// 4.3e-7 (1.2e-6); X times 2^-124 1.2e-7 (6.1e-7); one product alone 2.5e-8 (2.5e-8).
// Time, from a graph, against the 16-row tiles: 4096 x 4096 QT-P @ 4.25, M = 100, 120.8 -> 42.7 us; QT, M = 1024
// 565 -> 171, M = 2048 1128 -> 307 (224 TFLOP/s of fp32 results; the library's fp32 product 248 and 475 us). A K-step takes 1.9,
// 2.9 or 5.0 us at 32, 64 or 128 rows: decode and LDS stores, then the MFMAs (1.3 us at 64 rows), one after
// the other, as two buffers of three planes do not fit the LDS; the matrix pipes are busy 0.26 at M = 100.
#pragma once

enum { kXBf16, kXRound, kXSplit };   // X: bf16 / fp32 rounded to bf16 / fp32 cut into three planes

constexpr int kShortFlagBytes = 64;
constexpr float kPlaneScale = 0x1p24f;   // of X and the scales ahead of the planes (see above)

template <int XM, int TM>
struct ShortTile {
  static_assert(TM == 128 || TM == 64 || TM == 32, "row tiles of 128, 64 or 32 rows");
  static constexpr bool split = XM == kXSplit;
  // split: 1024 threads, but at 128 rows, where the two accumulators would leave them 64 registers for all else
  static constexpr int threads = split && TM < 128 ? 1024 : 512, waves = threads / 64;
  static constexpr int ct = kCells * 4 / threads;            // columns of a cell that one thread decodes
  static constexpr int planes = split ? 3 : 1;
  static constexpr int bufs = split ? 1 : 2;                 // LDS buffers of a step's tiles
  static constexpr int a_plane = TM * kTK * 2, b_plane = kTileBytes;
  static constexpr int buf_bytes = planes * (a_plane + b_plane);
  static constexpr int lds_bytes = bufs * buf_bytes + (split ? kShortFlagBytes : 0);
  static constexpr int ring = split && TM == 128 ? 2 : 4;    // register slots of cells (see step())
  static constexpr int xring = split ? 1 : 2;                // and of X segments
  // waves: wk along a step's rows of K (their sums are added at the end), wn across the columns, the rest down the rows
  static constexpr int wk = split && TM == 32 ? 2 : 1;
  static constexpr int wn = TM == 128 ? 4 : 8, wm = waves / wk / wn;
  static constexpr int ri = TM / 32 / wm, nj = 8 / wn;       // 32 x 32 tiles of a wave
  static constexpr int xrows = threads / 8;                  // X rows that one pass of the threads covers
  static constexpr int xsegs = TM > xrows ? TM / xrows : 1;  // 8-element X segments of a thread per step
};

// Upper halves of a (low) and b (high): two truncated bf16 values.
__device__ __forceinline__ uint32_t pack_hi(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float below_hi(float v) { return v - __uint_as_float(__float_as_uint(v) & 0xFFFF0000u); }

// Eight floats as three planes; with LO false the third is not formed (it is zero). nf turns NaN and
// stays so once a value is not finite (its remainder is NaN).
template <bool LO, bool CHECK>
__device__ __forceinline__ void split_planes(const float* v, u32x4_t& hi, u32x4_t& mid, u32x4_t& lo, float& nf) {
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const float a = v[2 * p], b = v[2 * p + 1];
    const float ra = below_hi(a), rb = below_hi(b);
    hi[p] = pack_hi(a, b);
    mid[p] = pack_hi(ra, rb);
    if constexpr (LO) lo[p] = pack_hi(below_hi(ra), below_hi(rb));
    if constexpr (CHECK) nf = __builtin_fmaf(ra, 0.0f, __builtin_fmaf(rb, 0.0f, nf));
  }
}

// decode_cell in fp32 for NC columns: out[j][r] = fma(u, s, -offset * s) for column j, row r, the exact W_hat value before
// any bf16 rounding. pw holds their 4 NC dwords (a class W4 cell's first NC, a W8 cell's first 2 NC).
template <bool PC, int NC>
__device__ __forceinline__ void decode_cols_f32(uint32_t cls, const uint32_t (&pw)[4 * NC], const float (&st)[NC],
                                                const float (&sb)[NC], float (&out)[NC][8]) {
  constexpr int NS = PC ? NC : 1;
  float ct[NS], cb[NS];
  auto offset_terms = [&](float off) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      ct[j] = -off * st[j];
      cb[j] = -off * sb[j];
    }
  };
  auto bytes = [&](int j, uint32_t top, uint32_t bot) __attribute__((always_inline)) {
    const int k = PC ? j : 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      out[j][r] = __builtin_fmaf((float)((top >> (8 * r)) & 0xFFu), st[k], ct[k]);
      out[j][4 + r] = __builtin_fmaf((float)((bot >> (8 * r)) & 0xFFu), sb[k], cb[k]);
    }
  };
  if (cls == 0) {
    offset_terms(8.0f);
#pragma unroll
    for (int j = 0; j < NC; ++j) bytes(j, opaque(pw[j] & 0x0F0F0F0Fu), opaque((pw[j] >> 4) & 0x0F0F0F0Fu));
  } else if (cls == 1) {
    offset_terms(128.0f);
#pragma unroll
    for (int j = 0; j < NC; ++j) bytes(j, pw[2 * j], pw[2 * j + 1]);
  } else if (cls == 2) {
    offset_terms(32768.0f);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int k = PC ? j : 0;
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const float s = h < 2 ? st[k] : sb[k], c = h < 2 ? ct[k] : cb[k];
        out[j][2 * h] = __builtin_fmaf((float)(pw[4 * j + h] & 0xFFFFu), s, c);
        out[j][2 * h + 1] = __builtin_fmaf((float)(pw[4 * j + h] >> 16), s, c);
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
      for (int r = 0; r < 8; ++r) out[j][r] = 0.0f;
  }
}

// A TM x 256 tile (rows m0.., columns of tile ct) of X * W_hat over K-steps kb0 .. kb0 + nks - 1 in plain fp32, each
// output a chain of fmas in K order: the path of a block that met a value that is not finite. Eight rows
// per thread at a time; thread t owns column t % 256 of the row groups t / 256, + NT / 256, ..
template <int kCF, int TM, int NT>
__device__ __forceinline__ void short_plain_f32(const mtc_tile_desc& d, const int ct, const int kb0, const int nks,
                                                const float* __restrict__ X, int64_t ldx, const int m0, const int M,
                                                float* __restrict__ y, int64_t ld, const int32_t* __restrict__ col_perm,
                                                unsigned char* lds) {
  constexpr int CW = cell_words(kCF);
  float* const wl = reinterpret_cast<float*>(lds);            // the step's W_hat, [64][256]
  const int t = threadIdx.x;
  const int n = ct * kTN + (t & (kTN - 1));
  for (int r0 = 0; r0 < TM; r0 += 8 * (NT / kTN)) {
    const int row0 = m0 + r0 + 8 * (t / kTN);
    const int rows = row0 < m0 + TM ? min(8, M - row0) : 0;
    float acc[8] = {};
    for (int ks = 0; ks < nks; ++ks) {
      const size_t step = (size_t)ct * d.n_ksteps + kb0 + ks;
      if (t < kCells) {
        const uint32_t* w = d.cells + (step * kCells + t) * CW;
        const uint32_t cls = (w[0] >> 14) & 3u, pos = (w[0] >> 16) & (kCells - 1);
        const uint32_t* src = d.payload + d.step_off[step] + (w[0] & 0x3FFFu);
        const int words = cls == 0 ? 4 : cls == 1 ? 8 : cls == 2 ? 16 : 0;
        for (int j = 0; j < 4; ++j) {
          uint32_t pw[4] = {};
          const int per = words / 4;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (i < per) pw[i] = src[per * j + i];
          const uint32_t sw = kCF == kCellCols ? w[1 + j] : w[1];
          const float st[1] = {kCF == kCellFp32 ? __uint_as_float(w[1]) : __uint_as_float(sw << 16)};
          const float sb[1] = {kCF == kCellFp32 ? __uint_as_float(w[2]) : __uint_as_float(sw & 0xFFFF0000u)};
          float o[1][8];
          decode_cols_f32<false, 1>(cls, pw, st, sb, o);
#pragma unroll
          for (int r = 0; r < 8; ++r) wl[(8 * (pos & 7u) + r) * kTN + 4 * (pos >> 3) + j] = o[0][r];
        }
      }
      __syncthreads();
      const int k0 = (kb0 + ks) * kTK, kn = min(kTK, d.K - k0);
      for (int k = 0; k < kn; ++k) {
        const float wv = wl[k * kTN + (t & (kTN - 1))];
#pragma unroll
        for (int r = 0; r < 8; ++r)
          if (r < rows) acc[r] = __builtin_fmaf(X[(int64_t)(row0 + r) * ldx + k0 + k], wv, acc[r]);
      }
      __syncthreads();
    }
    if (n < d.N) {
#pragma unroll
      for (int r = 0; r < 8; ++r)
        if (r < rows) y[(int64_t)(row0 + r) * ld + (col_perm ? col_perm[n] : n)] = acc[r];
    }
  }
}

// One TM-row output tile block of matrix `d` (arguments as gemm_tile_block).
template <int kCF, int kYDT, int XM, int TM>
__device__ __forceinline__ void gemm_short_block(const mtc_tile_desc& d, const int rt, const int ct, const int by,
                                                 const void* __restrict__ Xv, int64_t ldx, void* __restrict__ Y,
                                                 int64_t ldy, int M, int steps_per_split, float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  typedef ShortTile<XM, TM> T;
  constexpr int CW = cell_words(kCF), R = T::ring, NP = T::planes, NC = T::ct;
  constexpr bool PC = kCF == kCellCols;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = rt * TM, n0 = ct * kTN;
  const int kb0 = by * steps_per_split;
  const int nks = min(steps_per_split, d.n_ksteps - kb0);
  // words per cell of this stream (the kCellCols kernels also run bf16-pair members of a group or batch)
  const bool gcols = PC && (T::split || (d.flags & MTC_FLAG_COLS_GATHERED) != 0);
  const int cw = PC && !gcols ? 2 : CW;
  uint32_t* const flags = reinterpret_cast<uint32_t*>(lds + T::bufs * T::buf_bytes);   // split: [0..3] third weight
                                                                                       // plane of step i & 3, [4] plain
  // ---- cells: every load goes through a buffer resource, so that steps past the run and payload a class does
  // not have read zeros, and every thread issues the same loads whatever its cells
  const size_t step0 = (size_t)ct * d.n_ksteps + kb0;
  const __amdgpu_buffer_rsrc_t cell_r = buffer_of(d.cells + step0 * kCells * cw, (int64_t)nks * kCells * cw * 4);
  const __amdgpu_buffer_rsrc_t pay_r = buffer_of(d.payload, d.payload_dwords * 4);
  const uint32_t* step_off = d.step_off + step0;
  // slot: word 0 and the scale words of this thread's columns (one pair word, the two fp32 scales, or one word per
  // column of a gathered cell) and their payload but for the second half of P16 codes, loaded when they are decoded
  constexpr int SW = kCF == kCellBf16 ? 1 : kCF == kCellFp32 ? 2 : NC, NQ = NC / 2;
  uint32_t w[R], sc[R][SW], base[R];
  u32x4_t q[R][NQ];
  const int cell = tid / (4 / NC), cpart = tid % (4 / NC);   // columns cpart * NC .. of the cell
  // a gathered cell's scale words: with the descriptor, or with the payload where a whole cell's would take the
  // registers of a second slot (128-row tiles of fp32 results)
  constexpr bool kLateScales = PC && T::split && NC == 4;
  auto load_col_scales = [&](int i, int s) __attribute__((always_inline)) {
    const uint32_t so = (uint32_t)((i * kCells + cell) * cw) * 4u + 4u + (gcols ? 4u * NC * cpart : 0u);
    if constexpr (NC == 2) {
      const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(cell_r, so, 0, 0);
      sc[s][0] = v.x;
      sc[s][1] = v.y;
    } else {
      const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(cell_r, so, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) sc[s][SW == 4 ? j : 0] = v[j];
    }
  };
  auto load_desc = [&](int i, int s) __attribute__((always_inline)) {
    const uint32_t off = (uint32_t)((i * kCells + cell) * cw) * 4u;
    if constexpr (kCF == kCellBf16) {
      const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(cell_r, off, 0, 0);
      w[s] = v.x;
      sc[s][0] = v.y;
    } else if constexpr (kCF == kCellFp32) {
      const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(cell_r, off, 0, 0);
      w[s] = v.x;
      sc[s][0] = v.y;
      sc[s][1] = v.z;
    } else {
      w[s] = __builtin_amdgcn_raw_buffer_load_b32(cell_r, off, 0, 0);
      if constexpr (!kLateScales) load_col_scales(i, s);
    }
    base[s] = step_off[min(i, nks - 1)];
  };
  // bytes of this thread's columns in a cell of class cls: 4 NC, 8 NC or 16 NC
  auto payload_at = [&](int s, uint32_t cls) __attribute__((always_inline)) {
    return (base[s] + (w[s] & 0x3FFFu)) * 4u + (uint32_t)cpart * ((4u * NC) << (cls & 3u));
  };
  auto load_payload = [&](int i, int s) __attribute__((always_inline)) {
    if constexpr (kLateScales) load_col_scales(i, s);
    const uint32_t cls = (w[s] >> 14) & 3u, o = payload_at(s, cls);
    q[s][0] = __builtin_amdgcn_raw_buffer_load_b128(pay_r, cls < 3 ? o : kOutOfRange, 0, 0);
    if constexpr (NQ == 2)
      q[s][1] = __builtin_amdgcn_raw_buffer_load_b128(pay_r, cls == 1 || cls == 2 ? o + 16u : kOutOfRange, 0, 0);
  };
  // ---- X: segment tid % 8 (8 elements) of rows tid / 8, + xrows, .. of the tile; zeros past M and K
  constexpr int XB = XM == kXBf16 ? 2 : 4;                   // bytes per element
  const unsigned char* xbase = reinterpret_cast<const unsigned char*>(Xv) + (int64_t)m0 * ldx * XB;
  const __amdgpu_buffer_rsrc_t x_r =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(xbase), (short)0,
                                        (int)(uint32_t)min((int64_t)TM * ldx * XB, (int64_t)kOutOfRange), 0x00020000);
  const int xrow = tid >> 3, xseg = tid & 7;
  typedef u32x4_t XRegs[T::xsegs][XM == kXBf16 ? 1 : 2];
  XRegs xr[T::xring];
  auto load_x = [&](int i, XRegs& r) __attribute__((always_inline)) {
    const int k = (kb0 + i) * kTK + 8 * xseg;
#pragma unroll
    for (int h = 0; h < T::xsegs; ++h) {
      const int row = xrow + T::xrows * h;
      const bool in = row < TM && m0 + row < M && k < d.K && i < nks;
      const uint32_t off = in ? ((uint32_t)row * (uint32_t)ldx + (uint32_t)k) * (uint32_t)XB : kOutOfRange;
      r[h][0] = __builtin_amdgcn_raw_buffer_load_b128(x_r, off, 0, 0);
      if constexpr (XM != kXBf16) r[h][1] = __builtin_amdgcn_raw_buffer_load_b128(x_r, in ? off + 16u : kOutOfRange, 0, 0);
    }
  };
  float nf = 0.0f;                                           // NaN once a value was not finite (split)
  auto store_x = [&](unsigned char* as, const XRegs& r) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < T::xsegs; ++h) {
      const int row = xrow + T::xrows * h;
      if (TM < T::xrows && row >= TM) continue;
      unsigned char* const at = as + swz(row, xseg);
      if constexpr (XM == kXBf16) {
        *reinterpret_cast<u32x4_t*>(at) = r[h][0];
      } else {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = __uint_as_float(r[h][e >> 2][e & 3]);
        if constexpr (XM == kXRound) {
          *reinterpret_cast<u32x4_t*>(at) =
              u32x4_t{pk_bf16(v[0], v[1]), pk_bf16(v[2], v[3]), pk_bf16(v[4], v[5]), pk_bf16(v[6], v[7])};
        } else {
          u32x4_t p[3];
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] *= kPlaneScale;
          split_planes<true, true>(v, p[0], p[1], p[2], nf);
#pragma unroll
          for (int z = 0; z < 3; ++z) *reinterpret_cast<u32x4_t*>(at + z * T::a_plane) = p[z];
        }
      }
    }
  };
  uint32_t wide_pos = kCells;                                // position of this thread's P16 cell of the step, if it is one
  // ---- decode slot s into the B planes
  auto stage_cell = [&](unsigned char* bs, int s, int i) __attribute__((always_inline)) {
    const uint32_t cls = (w[s] >> 14) & 3u, pos = (w[s] >> 16) & (kCells - 1);
    uint32_t pw[4 * NC];
#pragma unroll
    for (int e = 0; e < 4 * NC; ++e) pw[e] = e < 4 * NQ ? q[s][e >> 2][e & 3] : 0u;
    const bool wide = __builtin_amdgcn_ballot_w64(cls == 2) != 0;
    if (wide) {                                              // P16 cells (rare): the other half of their codes
      const uint32_t o = payload_at(s, cls);
#pragma unroll
      for (int h = NQ; h < NC; ++h) {
        const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(pay_r, cls == 2 ? o + 16u * h : kOutOfRange, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) pw[4 * h + e] = v[e];
      }
      // waited for here: a wait after the branch would hold for the path without these loads too, and
      // there wait for every load sent ahead for the next steps
      __builtin_amdgcn_s_waitcnt(0x0F70);                    // vmcnt(0)
    }
    float st[NC], sb[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      if constexpr (kCF == kCellFp32) {
        st[j] = __uint_as_float(sc[s][0]);
        sb[j] = __uint_as_float(sc[s][1]);
      } else {
        const uint32_t first = sc[s][0], own = sc[s][PC ? j : 0];
        const uint32_t v = gcols ? own : first;
        st[j] = __uint_as_float(v << 16);
        sb[j] = __uint_as_float(v & 0xFFFF0000u);
      }
    }
    if constexpr (T::split) {
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        st[j] *= kPlaneScale;
        sb[j] *= kPlaneScale;
      }
    }
    const int col = (int)(pos >> 3) * 4 + cpart * NC, seg = (int)(pos & 7u);
    if constexpr (!T::split) {
      float o[NC][8];
      decode_cols_f32<PC, NC>(cls, pw, st, sb, o);
#pragma unroll
      for (int j = 0; j < NC; ++j)
        *reinterpret_cast<u32x4_t*>(bs + swz(col + j, seg)) = u32x4_t{
            pk_bf16(o[j][0], o[j][1]), pk_bf16(o[j][2], o[j][3]), pk_bf16(o[j][4], o[j][5]), pk_bf16(o[j][6], o[j][7])};
    } else {
      const float off = cls == 0 ? 8.0f : cls == 1 ? 128.0f : 32768.0f;
#pragma unroll
      for (int j = 0; j < (PC ? NC : 1); ++j)                // scales that are not finite, or overflow a code
        nf = __builtin_fmaf(off * st[j], 0.0f, __builtin_fmaf(off * sb[j], 0.0f, nf));
      constexpr bool LO = kCF == kCellFp32;
      if (!LO && wide && lane == 0) flags[i & 3] = 1u;
      wide_pos = !LO && cls == 2 ? pos : kCells;
      // two columns at a time: all four of a whole cell at once take registers that the sums need
#pragma unroll
      for (int j2 = 0; j2 < NC; j2 += 2) {
        uint32_t pw2[8];                                     // their dwords: from 1, 2 or 4 times j2 on
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          pw2[e] = pw[4 * j2 + e];
          if (j2 > 0 && e < 4) pw2[e] = cls == 1 ? pw[2 * j2 + e] : pw2[e];
          if (j2 > 0 && e < 2) pw2[e] = cls == 0 ? pw[j2 + e] : pw2[e];
        }
        const float st2[2] = {st[j2], st[j2 + 1]}, sb2[2] = {sb[j2], sb[j2 + 1]};
        float o[2][8];
        decode_cols_f32<PC, 2>(cls, pw2, st2, sb2, o);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          u32x4_t p[3];
          unsigned char* const at = bs + swz(col + j2 + j, seg);
          split_planes<LO, false>(o[j], p[0], p[1], p[2], nf);
          *reinterpret_cast<u32x4_t*>(at) = p[0];
          *reinterpret_cast<u32x4_t*>(at + T::b_plane) = p[1];
          if constexpr (LO) *reinterpret_cast<u32x4_t*>(at + 2 * T::b_plane) = p[2];
        }
        if (!LO && wide) {                                   // P16 cells: the third plane (zeros elsewhere)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            u32x4_t p[3];
            split_planes<true, false>(o[j], p[0], p[1], p[2], nf);
            if (cls == 2) *reinterpret_cast<u32x4_t*>(bs + 2 * T::b_plane + swz(col + j2 + j, seg)) = p[2];
          }
        }
        if constexpr (NC > 2) __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // ---- the step's MFMAs
  const int wn = wave % T::wn, wm = wave / T::wn % T::wm, wk = wave / (T::wn * T::wm);
  f32x16_t acc[T::ri][T::nj];
#pragma unroll
  for (int i = 0; i < T::ri; ++i)
#pragma unroll
    for (int j = 0; j < T::nj; ++j) acc[i][j] = f32x16_t{};
  f32x16_t low[T::split ? T::ri : 1][T::split ? T::nj : 1];
  if constexpr (T::split) {
#pragma unroll
    for (int i = 0; i < T::ri; ++i)
#pragma unroll
      for (int j = 0; j < T::nj; ++j) low[i][j] = f32x16_t{};
  }
  // (low: the sums of all plane pairs but the first)
  const int arow = wm * 32 * T::ri + (lane & 31), bcol = wn * 32 * T::nj + (lane & 31);
  // Operand addresses within a plane: 16-row slice kk of the step flips bits 1 and 2 of the segment, 32 more rows are
  // 4 KiB on (swz). Formed for each slice from one register a tile: kept for all slices they cost spills.
  constexpr int KK = kTK / 16 / T::wk;                       // 16-row slices of this wave
  const uint32_t a_at0 = swz(arow, wk * KK * 2 + (lane >> 5)), b_at0 = swz(bcol, wk * KK * 2 + (lane >> 5));
  auto frag = [&](const unsigned char* plane, uint32_t at, int t) __attribute__((always_inline)) {
    return *reinterpret_cast<const bf16x8_t*>(plane + at + t * 32 * 128);
  };
  auto mfma_step = [&](const unsigned char* as, const unsigned char* bs, bool third) __attribute__((always_inline)) {
    uint32_t a_at = a_at0, b_at = b_at0;
    if constexpr (T::split) asm volatile("" : "+v"(a_at), "+v"(b_at));
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const uint32_t ao = a_at ^ (uint32_t)(kk << 5), bo = b_at ^ (uint32_t)(kk << 5);
      bf16x8_t a[NP][T::ri], b[T::split ? 2 : 1][T::nj];
#pragma unroll
      for (int z = 0; z < (T::split ? 2 : 1); ++z)
#pragma unroll
        for (int j = 0; j < T::nj; ++j) b[z][j] = frag(bs + z * T::b_plane, bo, j);
#pragma unroll
      for (int i = 0; i < T::ri; ++i) {
#pragma unroll
        for (int z = 0; z < NP; ++z) a[z][i] = frag(as + z * T::a_plane, ao, i);
        auto products = [&](f32x16_t (&c)[T::ri][T::nj], int zb, int za) __attribute__((always_inline)) {
#pragma unroll
          for (int j = 0; j < T::nj; ++j)
            c[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[za][i], b[zb][j], c[i][j], 0, 0, 0);
        };
        if constexpr (T::split) {
          products(low, 1, 2);
          products(acc, 0, 0);
          products(low, 1, 1);
          products(low, 0, 2);
          products(low, 1, 0);
          products(low, 0, 1);
          __builtin_amdgcn_sched_barrier(0);                 // one slice's operands in registers at a time
        } else {
          products(acc, 0, 0);
        }
      }
    }
    if constexpr (T::split) if (third) {                     // the weights' third plane . X's first two
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        const uint32_t ao = a_at ^ (uint32_t)(kk << 5), bo = b_at ^ (uint32_t)(kk << 5);
#pragma unroll
        for (int i = 0; i < T::ri; ++i) {
          const bf16x8_t a1 = frag(as + T::a_plane, ao, i), a0 = frag(as, ao, i);
#pragma unroll
          for (int j = 0; j < T::nj; ++j) {
            const bf16x8_t b2 = frag(bs + 2 * T::b_plane, bo, j);
            low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b2, low[i][j], 0, 0, 0);
            low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b2, low[i][j], 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  // ---- Step i decodes slot i % R while the payloads of steps i + 1 .. i + R - 2 are in flight, then refills its
  // slot with the descriptors of step i + R and sends for the payload of step i + R - 1.
  auto step = [&](int i, int s, XRegs& x) __attribute__((always_inline)) {
    unsigned char* const as = lds + (T::bufs == 2 ? (i & 1) * T::buf_bytes : 0);
    unsigned char* const bs = as + NP * T::a_plane;
    if constexpr (T::split && TM == 128) {                   // X first: the decode then takes its registers
      store_x(as, x);
      __builtin_amdgcn_sched_barrier(0);
    }
    stage_cell(bs, s, i);
    if constexpr (!(T::split && TM == 128)) store_x(as, x);
    load_x(i + T::xring, x);                                 // first: loads return in order, and the next step waits for X
    load_desc(i + R, s);
    load_payload(i + R - 1, (s + R - 1) % R);
    bool third = kCF == kCellFp32;
    if constexpr (T::split && kCF != kCellFp32) {
      if (tid == 0) flags[(i + 2) & 3] = 0u;
    }
    lds_barrier();
    if constexpr (T::split && kCF != kCellFp32) third = __builtin_amdgcn_readfirstlane(flags[i & 3]) != 0;
    mfma_step(as, bs, third);
    if (T::bufs == 1) lds_barrier();                         // the tiles are free for the next step
    if (T::split && kCF != kCellFp32 && third) {             // the third weight plane back to zeros
      if (wide_pos < kCells) {
#pragma unroll
        for (int j = 0; j < NC; ++j)
          *reinterpret_cast<u32x4_t*>(bs + 2 * T::b_plane + swz((int)(wide_pos >> 3) * 4 + cpart * NC + j, (int)(wide_pos & 7u))) =
              u32x4_t{0u, 0u, 0u, 0u};
      }
      lds_barrier();
    }
  };
  // the first step's payload ahead of the later steps' descriptors, which would queue in front of it
  load_desc(0, 0);
  load_x(0, xr[0]);
#pragma unroll
  for (int s = 1; s < R; ++s) {
    load_desc(s, s);
    load_payload(s - 1, s - 1);
    if (s == 1 && T::xring == 2) load_x(1, xr[T::xring - 1]);
  }
  if (T::split) {                                            // (while the first loads are in flight)
    if (tid < 5) flags[tid] = 0u;
    unsigned char* const third_plane = lds + NP * T::a_plane + 2 * T::b_plane;
#pragma unroll
    for (int z = 0; z < T::b_plane / (16 * T::threads); ++z)
      *reinterpret_cast<u32x4_t*>(third_plane + (z * T::threads + tid) * 16) = u32x4_t{0u, 0u, 0u, 0u};
    lds_barrier();
  }
  static_assert(R % T::xring == 0, "the X registers' ring divides the cells'");
  for (int i0 = 0; i0 < nks; i0 += R) {
#pragma unroll
    for (int s = 0; s < R; ++s)
      if (i0 + s < nks) step(i0 + s, s, xr[s % T::xring]);
  }

  // ---- epilogue: C element e of lane l is row (e/4)*8 + (l/32)*4 + e%4, column l%32 (as gemm_tile_block)
  float* const yf = part ? part + (size_t)by * M * d.N : reinterpret_cast<float*>(Y);
  const int64_t ld = part ? (int64_t)d.N : ldy;
  const bool fp32_out = part || kYDT == MTC_DTYPE_F32;
  if constexpr (T::split) {
#pragma unroll
    for (int i = 0; i < T::ri; ++i)
#pragma unroll
      for (int j = 0; j < T::nj; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          acc[i][j][e] += low[i][j][e];
          nf = __builtin_fmaf(acc[i][j][e], 0.0f, nf);
          acc[i][j][e] *= 1.0f / (kPlaneScale * kPlaneScale);
        }
    if (nf != nf) flags[4] = 1u;
    __syncthreads();
    if (flags[4]) {
      __syncthreads();
      short_plain_f32<kCF, TM, T::threads>(d, ct, kb0, nks, reinterpret_cast<const float*>(Xv), ldx, m0, M, yf, ld,
                               part ? nullptr : d.col_perm, lds);
      return;
    }
  }
  if constexpr (T::wk == 2) {                                // add the two K halves
    static_assert(T::ri == 1 && T::nj == 1, "one 32 x 32 tile per wave");
    __syncthreads();
    float* const half = reinterpret_cast<float*>(lds) + (wave % T::wn) * 1024 + lane * 4;
    if (wk == 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<f32x4_t*>(half + 256 * e) =
            f32x4_t{acc[0][0][4 * e], acc[0][0][4 * e + 1], acc[0][0][4 * e + 2], acc[0][0][4 * e + 3]};
    }
    __syncthreads();
    if (wk == 1) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(half + 256 * e);
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[0][0][4 * e + c] += v[c];
    }
  }
#pragma unroll
  for (int j = 0; j < T::nj; ++j) {
    const int col = n0 + bcol + j * 32;
    if (col >= d.N) continue;
    const int ycol = (d.col_perm && !part) ? d.col_perm[col] : col;
#pragma unroll
    for (int i = 0; i < T::ri; ++i) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = m0 + wm * 32 * T::ri + i * 32 + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3);
        if (row < M) {
          if (fp32_out)
            yf[(int64_t)row * ld + ycol] = acc[i][j][e];
          else
            reinterpret_cast<__bf16*>(Y)[(int64_t)row * ldy + ycol] = (__bf16)acc[i][j][e];
        }
      }
    }
  }
}
