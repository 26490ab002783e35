// flex_tile.hip -- the MFMA tile kernel for contractions whose 256 x 256 tiles
// leave CUs idle or mostly padding: 64 x 64, 64 x 128 or 128 x 128 tiles (rows
// of X by MFMA rows: the columns of the GEMM, or the gate and up columns of the
// SwiGLU), several workgroups per CU, any K, any alignment of X, of Y and of
// row-major weights.
//
// Device time of the launches, weights from HBM, M x K x N, with the other
// kernels and with this one as dispatched: GEMM 4062 x 546 x 944 24.6 -> 12.6 us
// (one launch of 128 x 128 tiles for a padded copy of X and 64 workgroups of 256
// x 256 tiles), SwiGLU 411 x 896 x 4432 20.8 -> 13.4 us (one launch), SwiGLU 300 x
// 1000 x 1100 23.8 -> 15.4 us and GEMM 391 x 1440 x 2574 27.2 -> 20.0 us (four k
// splits, as many as before, without the padded copy; the first unsplit, with
// longer sums: 8.3 us).  Where 256 x 256 tiles fill the chip they stay ahead
// (GEMM 4096^3: 98 us against 139 us here): a 128 x 128 tile moves twice the
// operand bytes per multiply-add.
//
// Every operand goes memory -> registers -> LDS: a register load takes any
// 2-byte aligned address, where an LDS-DMA load needs aligned rows, and the
// compiler places its waits.  (X straight from memory into MFMA operands, 16
// rows x 64 bytes a load, was slower: half lines, and at a power-of-two row
// stride one L1 set -- GEMM 4096^3 187 us, 119 us without those loads.)  The
// loads run D steps ahead in registers; more steps than two or three cost the
// second (third, fourth) workgroup of a CU, which hides more than they do: D =
// 3 at one workgroup per CU 170 us, D = 2 at two 142 us.  Ring writes, operand
// reads and loads are spread over the MFMAs (sched_group_barrier), with one
// barrier per step between its halves.
//
// The sums are the tile kernel's own -- v_mfma_f32_16x16x32_bf16 over k in
// order -- so results equal its results at the same k split bit for bit.
#include <type_traits>

#include "common.h"
#include "launch.h"
#include "tile_ops.h"

namespace llk_gfx950 {

struct FlexArgs {
  const uint16_t* x;  // [M, K] bf16, row stride ldx (any alignment)
  const uint8_t* w0;  // packed payload (Wg, or B of the GEMM); RM: bf16 [K, N]
  const uint8_t* w1;  // Wu (SwiGLU)
  void* y;            // [M, N], row stride ldy (any alignment)
  float* part;        // [S][NMAT][M][n_pad] fp32 planes (S > 1)
  int64_t ldx, ldy, ldw0, ldw1;
  int M, N, K;
  int KB;             // ceil(K / 64)
  int tiles_m, tiles_n, group_m;
  int S, kbs, n_pad;
  int out, accumulate;
};

// Tile geometry: WM x WN waves, each MI x NI MFMA blocks of 16 x 16.
template <int NMAT, int WM, int MI, int NI>
struct FlexCfg {
  static constexpr int WN = 4 / WM;
  static constexpr int TM = 16 * WM * MI;           // rows of X
  static constexpr int TN = 16 * WN * NI;           // MFMA rows (columns of the matrices together)
  static constexpr int COLS = TN / NMAT;            // columns of Y
  static constexpr int WCOLS = COLS / WN;           // columns of Y per wave
  static constexpr int XOFF = TN * 128;             // X behind the weights in a slot
  static constexpr int SLOT = (TN + TM) * 128;      // one 64-k step
  static constexpr int XL = TM / 32;                // 16-byte loads of X per thread and step
  static constexpr int WL = TN / 32;                // of W
  static constexpr int ROWB = WCOLS * 4 + 16;       // epilogue staging row
  // 64-k steps of loads in flight, in registers
  static constexpr int D = MI * NI <= 4 ? 3 : 2;
  // waves per SIMD (= workgroups per CU) the registers are kept to
  static constexpr int waves(bool rm) { return MI * NI <= 4 ? (rm ? 3 : 4) : MI * NI <= 8 ? 3 : 2; }
  static constexpr int LDS = 2 * SLOT > 64 * ROWB ? 2 * SLOT : 64 * ROWB;
  static_assert(TM % 32 == 0 && TN % 32 == 0 && NI % NMAT == 0 && LDS <= 65536, "tile");
};

template <int NMAT, int WM, int MI, int NI, bool SPLIT, bool RM>
__global__ __launch_bounds__(256, (FlexCfg<NMAT, WM, MI, NI>::waves(RM))) void flex_tile_kernel(FlexArgs a) {
  using C = FlexCfg<NMAT, WM, MI, NI>;
  constexpr int NB = NI / NMAT;  // 16-column blocks of Y per wave
  constexpr int XL = C::XL, WL = C::WL;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;

  const int tiles = a.tiles_m * a.tiles_n;
  const int idx = xcd_remap(blockIdx.x, tiles * (SPLIT ? a.S : 1));
  const int split = SPLIT ? idx / tiles : 0;
  const int tile = idx - split * tiles;
  int tm, tn;
  {
    const int span = a.group_m * a.tiles_n;
    const int g = tile / span, r = tile - g * span;
    const int gm = min(a.group_m, a.tiles_m - g * a.group_m);
    tm = g * a.group_m + r % gm;
    tn = r / gm;
  }
  const int kb0 = SPLIT ? split * a.kbs : 0;
  const int nkb = SPLIT ? min(a.KB - kb0, a.kbs) : a.KB;
  const int m0 = tm * C::TM, n0 = tn * C::COLS;

  // ---- X: rows of 128 bytes per 64-k step, 16-byte chunk c of row r at
  // c ^ ((r >> 1) & 7); thread t moves chunk t % 8 of rows t / 8 + 32 q.
  // Rows past M re-read the last one (their results are never stored).
  const uint16_t* const xbase = a.x + (int64_t)m0 * a.ldx + (int64_t)kb0 * 64;
  uint32_t xoff[XL];  // bytes from xbase
#pragma unroll
  for (int q = 0; q < XL; ++q)
    xoff[q] = (uint32_t)min(32 * q + (tid >> 3), a.M - 1 - m0) * (uint32_t)(a.ldx * 2) + 16 * (tid & 7);
  const uint32_t xlds =
      (uint32_t)(C::XOFF + (tid >> 3) * 128 + (((tid & 7) ^ ((tid >> 4) & 7)) * 16));
  // A step that K ends inside (its index `tail`): each 16-byte chunk is read
  // at most up to column K, `xback` bytes early, and put right in LDS.
  const int kend = a.K - kb0 * 64;
  const int tail = kend / 64;
  const int xover = (tail * 64 + 8 * (tid & 7) + 8 - kend) * 2;  // > 0: past K
  const uint32_t xback = xover > 0 ? (uint32_t)xover : 0u;
  auto load_x = [&](int kb, u32x4 (&xr)[XL]) {
    const uint8_t* const p = reinterpret_cast<const uint8_t*>(xbase + (int64_t)kb * 64);
    const uint32_t back = xback & (kb == tail ? ~0u : 0u);
#pragma unroll
    for (int q = 0; q < XL; ++q) xr[q] = load16_any(p + (int64_t)(xoff[q] - (uint64_t)back));
  };
  auto load_x_part = [&](int kb, u32x4 (&xr)[XL]) {
    const int left = a.K - ((kb0 + kb) * 64 + 8 * (tid & 7));
    const uint8_t* const p = reinterpret_cast<const uint8_t*>(xbase + (int64_t)kb * 64);
#pragma unroll
    for (int q = 0; q < XL; ++q)
      xr[q] = load16_part(reinterpret_cast<const uint16_t*>(p + xoff[q]), left);
  };

  // ---- W.  Packed: operand o = 2 i + h (16 MFMA rows i of the tile, k half
  // h) is 1 KiB in the MFMA's lane order, four 256-byte runs of the payload;
  // wave w moves operands w, w + 4, ...  Row-major: slab p holds the tile's
  // MFMA rows 64 p .. (the SwiGLU's gate columns, then its up columns) as 64
  // k rows of 128 bytes, 16-byte chunk c of row r at c ^ sw(r), sw(r) =
  // 2 (bit 1 of r + 2 bit 3 of r): the eight 32-byte row pieces that a half
  // wave's transposed read names (rows 0..3 and 8..11) then cover the 64
  // banks once.  Load q brings rows 32 (q & 1) + t / 8 of slab q / 2.
  const uint8_t* wbase[WL];  // packed: wave-uniform
  uint32_t woff[WL], wlds[WL];
  int wcols[WL];             // row-major: columns from the chunk's first to N
#pragma unroll
  for (int q = 0; q < WL; ++q) {
    if constexpr (!RM) {
      const int o = q * 4 + wave, i = o >> 1, h = o & 1;
      const int mat = NMAT == 2 && i >= C::COLS / 16 ? 1 : 0;
      const int c = n0 + 16 * (i - mat * (C::COLS / 16));  // first column of the block
      const int nb = min(c >> 7, (a.n_pad >> 7) - 1);
      wbase[q] = (mat ? a.w1 : a.w0) + ((int64_t)nb * a.KB + kb0) * kBlockBytes +
                 (8 * h + ((c >> 5) & 3)) * kSubBytes + ((c >> 4) & 1) * 256;
      woff[q] = (uint32_t)((lane >> 5) * 4 * kSubBytes +
                           ((lane & 15) + 32 * ((lane >> 4) & 1)) * 16);
      wlds[q] = (uint32_t)(o * 1024 + lane * 16);
      wcols[q] = 0;
    } else {
      const int p = q >> 1, r = 32 * (q & 1) + (tid >> 3), c = tid & 7;
      const int row = 64 * p + 8 * c;  // MFMA row of the chunk
      const bool up = NMAT == 2 && row >= C::COLS;
      int col = n0 + (up ? row - C::COLS : row);
      if (col >= a.N) col = n0;  // columns that are never stored: any readable ones
      const int64_t ldw = up ? a.ldw1 : a.ldw0;
      wbase[q] = (up ? a.w1 : a.w0) + (((int64_t)kb0 * 64 + r) * ldw + col) * 2;
      woff[q] = (uint32_t)(128 * ldw);  // one step
      wlds[q] = (uint32_t)(p * 8192 + r * 128 + ((c ^ (2 * (((r >> 1) & 1) | ((r >> 2) & 2)))) * 16));
      wcols[q] = a.N - col;
    }
  }
  auto load_w = [&](int kb, u32x4 (&wr)[WL]) {
#pragma unroll
    for (int q = 0; q < WL; ++q) {
      if constexpr (!RM)
        wr[q] = *reinterpret_cast<const u32x4*>(wbase[q] + (int64_t)kb * kBlockBytes + woff[q]);
      else
        wr[q] = load16_any(wbase[q] + (int64_t)kb * woff[q]);
    }
  };
  // The split's last step where it reaches K: rows past K are zero, and the
  // last row is read no further than column N.
  auto load_w_part = [&](int kb, u32x4 (&wr)[WL]) {
    if constexpr (!RM) {
      load_w(kb, wr);
    } else {
#pragma unroll
      for (int q = 0; q < WL; ++q)
        wr[q] = load16_part(
            reinterpret_cast<const uint16_t*>(wbase[q] + (int64_t)kb * woff[q]),
            (kb0 + kb) * 64 + 32 * (q & 1) + (tid >> 3) < a.K ? wcols[q] : 0);
    }
  };
  auto write_w = [&](int slot, const u32x4 (&wr)[WL]) {
#pragma unroll
    for (int q = 0; q < WL; ++q)
      *reinterpret_cast<u32x4*>(smem + slot * C::SLOT + wlds[q]) = wr[q];
  };
  auto write_x = [&](int slot, const u32x4 (&xr)[XL]) {
#pragma unroll
    for (int q = 0; q < XL; ++q)
      *reinterpret_cast<u32x4*>(smem + slot * C::SLOT + xlds + q * 4096) = xr[q];
  };
  // A operand i of the wave, k half h.  Row-major: two transposed reads; the
  // group's lane 4 j + c names row 32 h + 8 (l / 16) + j (+ 4), columns
  // 16 q + 4 c of the slab.
  const int t_r = 8 * (lane >> 4) + ((lane >> 2) & 3), t_c = lane & 3;
  const int t_sw = ((t_r >> 1) & 1) | ((t_r >> 2) & 2);  // the same for t_r + 32 h, t_r + 4
  auto read_a = [&](const uint8_t* base, int i, int h) -> bf16x8 {
    const int blk = NMAT == 2 ? (i / NB) * (C::COLS / 16) + wn * NB + i % NB : wn * NI + i;
    if constexpr (!RM) {
      return *reinterpret_cast<const bf16x8*>(base + (2 * blk + h) * 1024 + lane * 16);
    } else {
      typedef short v4i16 __attribute__((ext_vector_type(4)));
      typedef __attribute__((address_space(3))) v4i16* lds_v4i16;
      const uint8_t* const p = base + (blk >> 2) * 8192 + h * 4096 + t_r * 128 +
                               ((blk & 3) ^ t_sw) * 32 + (t_c >> 1) * 16 + (t_c & 1) * 8;
      const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16)(p));
      const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16)(p + 512));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };
  // B operand j, k half h: row 16 (wm MI + j) + l % 16, chunk 4 h + l / 16.
  const int br = lane & 15;
  const uint32_t b_off[2] = {
      (uint32_t)(C::XOFF + (wm * MI * 16 + br) * 128 + (((lane >> 4) ^ (br >> 1)) * 16)),
      (uint32_t)(C::XOFF + (wm * MI * 16 + br) * 128 + (((4 + (lane >> 4)) ^ (br >> 1)) * 16))};

  f32x4 acc[NI][MI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  bf16x8 A[2][NI], B[2][MI];  // operands of the two k halves
  auto read_half = [&](int slot, int h) {
    const uint8_t* const base = smem + slot * C::SLOT;
#pragma unroll
    for (int j = 0; j < MI; ++j)
      B[h][j] = *reinterpret_cast<const bf16x8*>(base + b_off[h] + j * 2048);
#pragma unroll
    for (int i = 0; i < NI; ++i) A[h][i] = read_a(base, i, h);
  };
  auto mma_half = [&](int h) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < MI; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[h][i], B[h][j], acc[i][j], 0, 0, 0);
  };
  // One half step: its MFMAs with the other half's operand reads, `L` ring
  // writes and `L` loads spread between them.
  auto spread = [&](auto Lc) {
    constexpr int L = decltype(Lc)::value;
    constexpr int RD = MI + (RM ? 2 : 1) * NI, MM = MI * NI;
    constexpr int per = MM > RD + 2 * L ? MM / (RD + 2 * L) : 1;
#pragma unroll
    for (int r = 0; r < RD; ++r) {
      __builtin_amdgcn_sched_group_barrier(0x008, per, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
#pragma unroll
    for (int r = 0; r < L; ++r) {
      __builtin_amdgcn_sched_group_barrier(0x008, per, 0);
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
    }
#pragma unroll
    for (int r = 0; r < L; ++r) {
      __builtin_amdgcn_sched_group_barrier(0x008, per, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, MM, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // Whole 64-k steps, then the one K ends inside (row-major weights: the step
  // that holds the last row).
  //
  // Two LDS slots, one barrier per step, between its halves: the first half's
  // MFMAs cover the second half's operand reads, the second half's the next
  // step's.  Slot k & 1 is free after step k's barrier (all its operands are
  // read) and takes step k + 2: its weights in the second half of step k, its
  // X in the first half of step k + 1, both before that step's barrier.  The
  // registers a write frees are loaded again at once, D steps ahead.  Loads
  // past the end re-read the last step: a uniform count of loads per step
  // keeps the compiler's waits exact.
  const int nfull = min(nkb, (RM ? kend - 1 : kend) / 64);
  if (nfull > 0) {
    constexpr int D = C::D;
    u32x4 xr[D][XL], wr[D][WL];
    const bool in_ring = !RM && nfull < nkb;  // K ends inside step nfull
    const int last = in_ring ? nfull : nfull - 1;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      load_w(min(d, last), wr[d]);
      load_x(min(d, last), xr[d]);
    }
    write_w(0, wr[0]);
    load_w(min(D, last), wr[0]);
    write_x(0, xr[0]);
    load_x(min(D, last), xr[0]);
    __syncthreads();
    read_half(0, 0);
    write_w(1, wr[1]);
    load_w(min(D + 1, last), wr[1]);
    __builtin_amdgcn_sched_barrier(0);
    int kb = 0;
    auto step = [&](auto Uc) {
      constexpr int U = decltype(Uc)::value;
      const int slot = kb & 1;
      read_half(slot, 1);
      write_x(slot ^ 1, xr[(U + 1) % D]);
      load_x(min(kb + 1 + D, last), xr[(U + 1) % D]);
      mma_half(0);
      spread(std::integral_constant<int, XL>{});
      __syncthreads();
      read_half(slot ^ 1, 0);
      write_w(slot, wr[(U + 2) % D]);
      load_w(min(kb + 2 + D, last), wr[(U + 2) % D]);
      mma_half(1);
      spread(std::integral_constant<int, WL>{});
      ++kb;
    };
    using std::integral_constant;
    while (true) {
      step(integral_constant<int, 0>{});
      if (kb >= nfull) break;
      step(integral_constant<int, 1>{});
      if (kb >= nfull) break;
      if constexpr (D > 2) {
        step(integral_constant<int, 2>{});
        if (kb >= nfull) break;
      }
    }
    __syncthreads();  // the ring is free
    if (in_ring) {
      // Step nfull is in its slot as loaded: every thread moves its own
      // chunks of X `xback` bytes down, zeros after them.
      const int slot = nfull & 1, bits = 8 * (int)xback;
#pragma unroll
      for (int q = 0; q < XL; ++q) {
        uint64_t* const p = reinterpret_cast<uint64_t*>(smem + slot * C::SLOT + xlds + q * 4096);
        const uint64_t lo = p[0], hi = p[1];
        if (bits >= 64) {
          p[0] = bits >= 128 ? 0 : hi >> (bits - 64);
          p[1] = 0;
        } else if (bits > 0) {
          p[0] = (lo >> bits) | (hi << (64 - bits));
          p[1] = hi >> bits;
        }
      }
      __syncthreads();
      read_half(slot, 0);
      read_half(slot, 1);
      mma_half(0);
      mma_half(1);
      __syncthreads();
    }
  }
  if (nfull < nkb && (RM || nfull == 0)) {
    u32x4 xs[XL], ws[WL];
    load_w_part(nfull, ws);
    load_x_part(nfull, xs);
    write_w(0, ws);
    write_x(0, xs);
    __syncthreads();
    read_half(0, 0);
    read_half(0, 1);
    mma_half(0);
    mma_half(1);
    __syncthreads();
  }

  // ---- epilogue: acc[i][j] holds, in lane l, row 16 (wm MI + j) + l % 16 and
  // columns 16 i + 4 (l / 16) + 0..3 of the wave's.  Staged as fp32, 16 rows
  // at a time, in LDS of the wave's own, then moved as 16-byte chunks of rows.
  uint8_t* const stage = smem + wave * 16 * C::ROWB;
  const int h4 = 4 * (lane >> 4);
  const int nw = n0 + wn * C::WCOLS;
  auto sync_wave = [&]() {
    wait_lgkmcnt0();
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
  };
  constexpr int planes = NMAT == 2 && SPLIT ? 2 : 1;
#pragma unroll
  for (int j = 0; j < MI; ++j) {
    const int mj = m0 + 16 * (wm * MI + j);
#pragma unroll
    for (int p = 0; p < planes; ++p) {
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        f32x4 v = acc[p * NB + i][j];
        if constexpr (NMAT == 2 && !SPLIT) {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = swiglu_act(acc[i][j][q], acc[NB + i][j][q]);
        }
        *reinterpret_cast<f32x4*>(stage + br * C::ROWB + (16 * i + h4) * 4) = v;
      }
      sync_wave();
      if (SPLIT || a.out == kOutF32) {
        float* const dst = SPLIT
            ? a.part + (((int64_t)split * NMAT + p) * a.M + mj) * a.n_pad + nw
            : static_cast<float*>(a.y) + (int64_t)mj * a.ldy + nw;
        const int64_t ld = SPLIT ? a.n_pad : a.ldy;
        const int cols_ok = (SPLIT ? a.n_pad : a.N) - nw;
        constexpr int CPR = C::WCOLS / 4;  // 16-byte chunks per row
#pragma unroll
        for (int q = 0; q < (16 * CPR + 63) / 64; ++q) {
          const int id = q * 64 + lane, row = id / CPR, c = (id % CPR) * 4;
          if (16 * CPR % 64 != 0 && id >= 16 * CPR) continue;
          if (mj + row >= a.M || c >= cols_ok) continue;
          f32x4 v = *reinterpret_cast<const f32x4*>(stage + row * C::ROWB + c * 4);
          float* const out = dst + row * ld + c;
          if (c + 4 <= cols_ok) {
            if (!SPLIT && NMAT == 1 && a.accumulate) v += __builtin_bit_cast(f32x4, load16_any(out));
            store16_any(out, __builtin_bit_cast(u32x4, v));
          } else {
            for (int e = 0; e < 4; ++e)
              if (c + e < cols_ok) out[e] = !SPLIT && NMAT == 1 && a.accumulate ? v[e] + out[e] : v[e];
          }
        }
      } else {
        uint16_t* const dst = static_cast<uint16_t*>(a.y) + (int64_t)mj * a.ldy + nw;
        const int cols_ok = a.N - nw;
        constexpr int CPR = C::WCOLS / 8;
        const bool f16 = a.out == kOutF16;
        auto widen = [&](uint16_t b) {
          return f16 ? (float)__builtin_bit_cast(_Float16, b) : bf16_bits_to_f32(b);
        };
#pragma unroll
        for (int q = 0; q < (16 * CPR + 63) / 64; ++q) {
          const int id = q * 64 + lane, row = id / CPR, c = (id % CPR) * 8;
          if (16 * CPR % 64 != 0 && id >= 16 * CPR) continue;
          if (mj + row >= a.M || c >= cols_ok) continue;
          const float* const src = reinterpret_cast<const float*>(stage + row * C::ROWB) + c;
          const f32x4 lo = *reinterpret_cast<const f32x4*>(src);
          const f32x4 hi = *reinterpret_cast<const f32x4*>(src + 4);
          uint16_t* const out = dst + row * a.ldy + c;
          float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          const bool full = c + 8 <= cols_ok;
          if (NMAT == 1 && a.accumulate) {
            const u32x4 old = full ? load16_any(out) : load16_part(out, cols_ok - c);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += widen((uint16_t)(old[e >> 1] >> (16 * (e & 1))));
          }
          u32x4 r;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            r[e] = f16 ? (uint32_t)f32_to_f16_rne(v[2 * e]) | ((uint32_t)f32_to_f16_rne(v[2 * e + 1]) << 16)
                       : f32x2_to_bf16x2_rne(v[2 * e], v[2 * e + 1]);
          if (full) {
            store16_any(out, r);
          } else {
            for (int e = 0; e < 8; ++e)
              if (c + e < cols_ok) out[e] = (uint16_t)(r[e >> 1] >> (16 * (e & 1)));
          }
        }
      }
      sync_wave();
    }
  }
}

template <int NMAT, int WM, int MI, int NI, bool SPLIT, bool RM>
const char* flex_tile_symbol() {
  static const std::string name = "_ZN10llk_gfx95016flex_tile_kernelI" + mangle_int(NMAT) +
                                  mangle_int(WM) + mangle_int(MI) + mangle_int(NI) + mangle_bool(SPLIT) + mangle_bool(RM) +
                                  "EEvNS_8FlexArgsE";
  return name.c_str();
}

template <int NMAT, int WM, int MI, int NI, bool SPLIT, bool RM>
static hipError_t launch_flex_t(FlexArgs& a, const llk::ModuleFns* mod, hipStream_t s) {
  auto fn = flex_tile_kernel<NMAT, WM, MI, NI, SPLIT, RM>;
  using C = FlexCfg<NMAT, WM, MI, NI>;
  a.tiles_m = (a.M + C::TM - 1) / C::TM;
  a.tiles_n = (a.N + C::COLS - 1) / C::COLS;
  a.group_m = 2048 / C::TM;
  return launch_kernel(mod, reinterpret_cast<const void*>(fn), &flex_tile_symbol<NMAT, WM, MI, NI, SPLIT, RM>,
                       dim3((unsigned)(a.tiles_m * a.tiles_n * a.S)), dim3(256), C::LDS, s, a);
}

template <int NMAT, int WM, int MI, int NI, bool RM>
static hipError_t launch_flex_s(FlexArgs& a, const llk::ModuleFns* mod, hipStream_t s) {
  return a.S > 1 ? launch_flex_t<NMAT, WM, MI, NI, true, RM>(a, mod, s)
                 : launch_flex_t<NMAT, WM, MI, NI, false, RM>(a, mod, s);
}

template <int NMAT>
static hipError_t launch_flex(FlexArgs& a, int cfg, bool rm, const llk::ModuleFns* mod,
                              hipStream_t s) {
  if (cfg == 222)
    return rm ? launch_flex_s<NMAT, 2, 2, 2, true>(a, mod, s)
              : launch_flex_s<NMAT, 2, 2, 2, false>(a, mod, s);
  if (cfg == 224)
    return rm ? launch_flex_s<NMAT, 2, 2, 4, true>(a, mod, s)
              : launch_flex_s<NMAT, 2, 2, 4, false>(a, mod, s);
  if (cfg == 244)
    return rm ? launch_flex_s<NMAT, 2, 4, 4, true>(a, mod, s)
              : launch_flex_s<NMAT, 2, 4, 4, false>(a, mod, s);
  return hipErrorInvalidValue;
}

}  // namespace llk_gfx950

// Whether the flex tile kernel takes M rows of X with row stride ldx (and
// row-major weights with row strides ldw0, ldw1; 0: packed): its byte
// offsets within a tile's rows of X and a step's rows of weights are 32-bit.
bool llk_flex_fits(int64_t M, int64_t K, int64_t ldx, int64_t ldw0, int64_t ldw1) {
  constexpr int64_t kMaxLd = (int64_t)1 << 24;
  return M >= 1 && M <= ((int64_t)1 << 30) && K >= 1 && K <= ((int64_t)1 << 30) && ldx < kMaxLd &&
         ldw0 < kMaxLd && ldw1 < kMaxLd;
}

// Internal.  mode 1 = fused SwiGLU (w0 = Wg, w1 = Wu; bf16 or fp32 y), 0 =
// GEMM (w0 = B; any y; with accumulate and S = 1 y += x w0).  cfg: the tile
// (222: 64 x 64, 224: 64 x 128, 244: 128 x 128 MFMA rows).  Weights packed, or
// with rowmajor bf16 [K, N] of row strides ldw0 / ldw1.  S > 1 leaves the fp32
// planes part[S][nmat][M][128 ceil(N / 128)] of the k split (every split
// non-empty) for llk_launch_split_reduce, which then applies the epilogue.
hipError_t llk_launch_flex(int mode, int cfg, const uint16_t* x, int64_t ldx, const void* w0,
                           int64_t ldw0, const void* w1, int64_t ldw1, void* y, int64_t ldy,
                           int M, int N, int K, int S, void* part, int out, bool accumulate,
                           bool rowmajor, const llk::ModuleFns* mod, hipStream_t s) {
  using namespace llk_gfx950;
  FlexArgs a{};
  a.x = x;
  a.w0 = static_cast<const uint8_t*>(w0);
  a.w1 = static_cast<const uint8_t*>(w1);
  a.y = y;
  a.part = static_cast<float*>(part);
  a.ldx = ldx;
  a.ldy = ldy;
  a.ldw0 = ldw0;
  a.ldw1 = ldw1;
  a.M = M;
  a.N = N;
  a.K = K;
  a.KB = (K + 63) / 64;
  a.S = S > 1 ? S : 1;
  a.kbs = (a.KB + a.S - 1) / a.S;
  a.n_pad = (N + kPackN - 1) / kPackN * kPackN;
  a.out = out;
  a.accumulate = accumulate ? 1 : 0;
  if (!llk_flex_fits(M, K, ldx, ldw0, ldw1) || N < 1 || (accumulate && mode != 0) ||
      (mode == 1 && out == kOutF16))
    return hipErrorInvalidValue;
  if (a.S > 1 && (part == nullptr || (int64_t)(a.S - 1) * a.kbs >= a.KB)) return hipErrorInvalidValue;
#if !defined(LLK_CO_OP) || LLK_CO_OP == 1
  if (mode == 1) return launch_flex<2>(a, cfg, rowmajor, mod, s);
#endif
#if !defined(LLK_CO_OP) || LLK_CO_OP == 0
  if (mode == 0) return launch_flex<1>(a, cfg, rowmajor, mod, s);
#endif
  return hipErrorInvalidValue;
}
