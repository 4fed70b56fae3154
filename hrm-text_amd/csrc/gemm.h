// Projection GEMMs of the HRM block with the RMSNorm before them and the SwiGLU after
// them fused in (models/transformer.py:87-92 pre-norm, models/layers.py:124-135 gqkv
// projection, :158-168 gate_up projection and SwiGLU).
//
//   y = rmsnorm(x) W^T                         (PLAIN: the attention's gqkv projection)
//   y = silu(rmsnorm(x) Wg^T) * (rmsnorm(x) Wu^T)   (SWIGLU: the MLP's gate_up + SwiGLU)
//
// x: bf16 [M, K] (row stride ldx), W: bf16 [N, K] (row stride ldw; for SWIGLU the first
// F rows are the gate, the next F rows the up projection, N = 2F), y: bf16 [M, Nout]
// (Nout = N, or F for SWIGLU). The weightless RMSNorm is a per-row scale,
// rmsnorm(x) W^T = diag(r) (x W^T) with r = (mean(x^2) + eps)^(-1/2), so the kernel
// multiplies x's raw rows (never writing the normalized x) and applies r, read from
// `rstd` (one fp32 per row, from a row pass before the GEMM; the kernel for few rows computes
// and writes it itself), to the fp32 products.
// With norm off, r = 1. Each output is rounded to bf16 once.
//
// Workgroup: MT x rows by 256 W rows, 8 waves (two per SIMD) of MT / 2 x rows by 64 W rows,
// K in stages of 64 staged by direct global->LDS loads (two stages: the next one lands
// while this one is read). Every wave computes Y^T tiles (A = W rows, B = x rows; lane =
// output row, registers = output columns), so a gate tile and its up tile meet in the
// same lanes and the epilogue stores whole rows.
//
// Persistent: one workgroup per CU walks its tiles, and the stages of successive tiles form
// one stream, so the next tile's first stages load under this tile's last ones and its
// epilogue (which stages through LDS of its own).
//
// Bound by the board's power at large M (a stage takes the same 2700 cycles at any load, at
// 2.4 GHz for 44 workgroups and about 1.75 with every CU busy), by the fill of the CUs at small
// M. K 2048, N 11264 with SwiGLU, the norm's pass included: M 16384 615 us (1.23 PFLOP/s; 609 to
// 634 on different cards), M 1100 55 us. A workgroup per tile, m tiles dealt to the XCDs by number
// and a stage's direct loads issued in one burst took 2% more and twice as long: five m tiles kept
// three XCDs idle and gave the others two rounds.
#pragma once
#include "common.h"

namespace prefixlm {
namespace mlp {

constexpr int WT = 256;              // W rows per workgroup
constexpr int KT = 64;               // K per stage (four MFMA k steps between barriers)
constexpr int KS = KT / 16;          // MFMA k steps per stage
constexpr int NTH = 512;             // 8 waves, two per SIMD
constexpr int ROWB = KT * 2;         // bytes of one staged row
constexpr int CPR = ROWB / 16;       // 16-byte chunks per staged row
constexpr int OUT_ROW = 64 * 2;      // output staging row: 64 bf16, chunks swizzled

template <int MT>
struct Geo {
  static constexpr int MI = MT / 64;             // 32-row x operands per wave
  static constexpr int NX = MT / 64;             // direct x loads per wave and stage (8 rows each)
  static constexpr int NW = WT / 64;             // direct W loads per wave and stage
  static constexpr int A_BYTES = MT * ROWB;      // x tile
  static constexpr int STAGE = A_BYTES + WT * ROWB;
  static constexpr int OUT = 2 * STAGE;          // output staging, 32 rows per wave
  static constexpr int LDS_BYTES = OUT + 8 * 32 * OUT_ROW;
  static_assert(KS == 4 && CPR == 8 && NX <= NW && LDS_BYTES <= 160 * 1024, "stage geometry");
};

// Staged row r, logical 16-byte chunk c lives at r * ROWB + 16 (c ^ f(r)), f(r) = (r / 2) % 8:
// the 16 rows of one quarter-wave operand read (a fixed chunk) land on 16 different 16-byte
// positions of the 256-byte bank window, so the operand reads are free of bank conflicts.
__device__ __forceinline__ int swz_f(int r) { return (r >> 1) & 7; }

struct Params {
  const bf16* x;
  const bf16* w;
  bf16* y;
  const float* rstd;   // [M] row scales (NORM)
  int64_t ldx, ldw, ldy;
  int M, K, N;       // N: W rows (2F for SWIGLU)
  int m_tiles, n_tiles;
};

// Tile number -> (m tile, n tile): groups of 8 m tiles, n after n within a group, so the 32
// consecutive tiles that an XCD's CUs work on together share 8 x slices and 4 W slices in its L2.
__device__ __forceinline__ void tile_at(const Params& P, int id, int* mt, int* nt) {
  const int per = 8 * P.n_tiles, g = id / per, r = id - g * per;
  const int gm = min(8, P.m_tiles - 8 * g);
  *nt = r / gm;
  *mt = 8 * g + (r - *nt * gm);
}

// 16 bytes per lane straight to LDS, lane j at dst + 16 j (dst wave-uniform)
typedef __attribute__((address_space(3))) char lds_char;
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t rsrc, lds_char* dst, uint32_t voffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)dst, 16, voffset, 0, 0, 0);
}

template <int MT, bool SWIGLU, bool NORM>
__global__ __launch_bounds__(NTH, 1) void proj_gemm_kernel(Params P) {
  using G = Geo<MT>;
  constexpr int MI = G::MI;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // XCD b % 8 takes a contiguous eighth of the tiles, its workgroups one after another
  const int total = P.m_tiles * P.n_tiles, xcd = blockIdx.x & 7;
  const int t_end = (int)((int64_t)(xcd + 1) * total / 8), step = gridDim.x >> 3;
  int id = (int)((int64_t)xcd * total / 8) + (int)(blockIdx.x >> 3);
  if (id >= t_end) return;
  const int F = P.N >> 1;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wm = w >> 2, wn = w & 3;   // 2 x 4 waves

  // Direct global -> LDS loads: one instruction moves 8 rows (1 KB); lane L writes slot L % 8
  // of row L / 8, which holds logical chunk (L % 8) ^ f(row). Wave w loads x rows
  // MT / 8 * w .. and W rows 32 w .. of the tile (SWIGLU: waves 0-3 gate rows, 4-7 up rows).
  uint32_t xoff[G::NX], woff[G::NW];
#pragma unroll
  for (int i = 0; i < G::NX; ++i) {
    const int r = MT / 8 * w + 8 * i + lane / CPR;
    xoff[i] = (uint32_t)((int64_t)r * P.ldx * 2) + 16 * ((lane % CPR) ^ swz_f(r));
  }
#pragma unroll
  for (int i = 0; i < G::NW; ++i) {
    const int r = 32 * w + 8 * i + lane / CPR;
    const int row = SWIGLU && w >= 4 ? F + r - 128 : r;
    woff[i] = (uint32_t)((int64_t)row * P.ldw * 2) + 16 * ((lane % CPR) ^ swz_f(r));
  }
  const int nk = P.K / KT;
  int mt, nt;
  tile_at(P, id, &mt, &nt);
  // the load cursor: the stage after the last one issued; past the last tile it stays on that
  // tile's last stage (loads into buffers nobody reads, so that every stage issues the same)
  int ld_id = id, ld_kk = 0, ld_mt = mt, ld_nt = nt;
  auto advance = [&]() {
    if (ld_kk + 1 < nk) {
      ++ld_kk;
    } else if (ld_id + step < t_end) {
      ld_id += step;
      ld_kk = 0;
      tile_at(P, ld_id, &ld_mt, &ld_nt);
    }
  };
  // direct loads [lo, hi) of the cursor's stage into buffer buf
  auto issue = [&](int buf, int lo, int hi) {
    const uint32_t k2 = (uint32_t)(ld_kk * ROWB);
    // W rows of n tile nt: from row 128 nt of each half (SWIGLU) or 256 nt on
    const int m0 = ld_mt * MT, n0 = ld_nt * (SWIGLU ? WT / 2 : WT);
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(P.x + (int64_t)m0 * P.ldx, rows_bytes(min(MT, P.M - m0), P.ldx, P.K));
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(P.w + (int64_t)n0 * P.ldw, rows_bytes(P.N - n0, P.ldw, P.K));
    lds_char* base = (lds_char*)smem + buf * G::STAGE;
#pragma unroll
    for (int i = lo; i < hi; ++i) {
      if (i < G::NX) load_lds16(xr, base + MT / 8 * w * ROWB + 1024 * i, xoff[i] + k2);
      load_lds16(wr, base + G::A_BYTES + 32 * w * ROWB + 1024 * i, woff[i] + k2);
    }
  };

  // operand reads: A = W rows (lane = W row of the tile), B = x rows (lane = x row);
  // logical chunk 2 ks + hh of k step ks, at 16 ((2 ks + hh) ^ f(l32)) of the row (the
  // operand row bases are multiples of 32)
  int coff[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) coff[ks] = 16 * ((2 * ks + hh) ^ swz_f(l32));
  // W tile rows of A operand bi: SWIGLU: bi = 0 the gate rows 32 wn, bi = 1 the up rows
  // 128 + 32 wn of the same output columns; PLAIN: 64 wn + 32 bi
  auto a_row = [&](int bi) { return SWIGLU ? bi * (WT / 2) + 32 * wn : 64 * wn + 32 * bi; };
  const int brow0 = MT / 2 * wm;   // x rows of B operand mi: brow0 + 32 mi

  f32x16 acc[MI][2];   // [mi: x rows][bi: W rows]; Y^T tiles (register = W row, lane = x row)
  // LDS reads of k step ks of buffer buf into fragment set `set`
  bf16x8 af[2][2], bfr[2][MI];
  auto rd = [&](int buf, int ks, int set) {
    const char* abase = smem + buf * G::STAGE + G::A_BYTES + l32 * ROWB + coff[ks];
    const char* bbase = smem + buf * G::STAGE + l32 * ROWB + coff[ks];
#pragma unroll
    for (int i = 0; i < 2; ++i) af[set][i] = *reinterpret_cast<const bf16x8*>(abase + a_row(i) * ROWB);
#pragma unroll
    for (int i = 0; i < MI; ++i) bfr[set][i] = *reinterpret_cast<const bf16x8*>(bbase + (brow0 + 32 * i) * ROWB);
  };
  auto mm = [&](int set, int mi) {
#pragma unroll
    for (int bi = 0; bi < 2; ++bi) acc[mi][bi] = mfma32x32x16(af[set][bi], bfr[set][mi], acc[mi][bi]);
  };
  // waits until this wave's loads of the stage in flight are in LDS, then a plain barrier
  // (the workgroup fence of __syncthreads would also wait for the output stores)
  auto stage_barrier = [&]() {
    sched_fence();
    waitcnt<0, 0>();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    sched_fence();
  };

  // In the last k step of a stage, after its first MFMAs, the next stage is waited for, the
  // workgroup syncs, and the buffer of this stage (every wave's reads of it are done) takes
  // the stage after: half of its direct loads between this step's MFMAs and half between
  // those of the next stage's first step. All of them at once, before the operand reads, kept
  // the matrix cores idle while eight waves issued 64 KB.
  constexpr int HALF = G::NW / 2;
  issue(0, 0, G::NW);
  advance();
  stage_barrier();   // stage 0 in LDS
  issue(1, 0, HALF);
  rd(0, 0, 0);
  int buf = 0;
  for (;;) {
    const int m0 = mt * MT;
    float rs[MI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      rs[mi] = NORM ? P.rstd[min(m0 + brow0 + 32 * mi + l32, P.M - 1)] : 1.f;
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mi][bi][r] = 0.f;
    }
    for (int kk = 0; kk < nk; ++kk) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int set = ks & 1;
        sched_fence();
        mm(set, 0);
        sched_fence();
        if (ks + 1 < KS) {
          rd(buf, ks + 1, set ^ 1);
        } else {
          // this step's operands are in registers before the barrier after which other waves load
          // into this buffer: the branches of advance() end the block here, and the compiler would
          // otherwise move reads used only after them past the barrier
#pragma unroll
          for (int m = 1; m < MI; ++m) settle(__builtin_bit_cast(u32x4, bfr[set][m]));
          stage_barrier();
          advance();
          rd(buf ^ 1, 0, set ^ 1);
        }
#pragma unroll
        for (int m = 1; m < MI; ++m) {
          sched_fence();
          if (m <= HALF) {
            constexpr int PER = MI - 1 < HALF ? HALF : 1;   // loads per slot (MT 128: one slot)
            if (ks == KS - 1) issue(buf, PER * (m - 1), PER * m);
            if (ks == 0) issue(buf ^ 1, HALF + PER * (m - 1), HALF + PER * m);
          }
          sched_fence();
          mm(set, m);
        }
      }
      buf ^= 1;
    }
    // ---- epilogue ----------------------------------------------------------------
    // 32 rows at a time through the wave's own LDS (chunk c of row r at c ^ (r % 8)), stored
    // as whole rows of the wave's columns: 32 (SWIGLU) or 64
    char* wl = smem + G::OUT + w * 32 * OUT_ROW;
    constexpr int NOT = SWIGLU ? 1 : 2;                      // output 32-column tiles of the wave
    constexpr int CPO = 4 * NOT, RPP = 64 / CPO;             // 16-byte chunks per row, rows per pass
    const int ycol0 = SWIGLU ? nt * (WT / 2) + 32 * wn : nt * WT + 64 * wn;
    const __amdgpu_buffer_rsrc_t yr = make_rsrc(P.y + (int64_t)m0 * P.ldy,
                                                rows_bytes(min(MT, P.M - m0), P.ldy, SWIGLU ? F : P.N));
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      // lane holds columns 8 (reg / 4) + 4 hh + reg % 4 of each 32-column tile
#pragma unroll
      for (int ti = 0; ti < NOT; ++ti)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float o[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (SWIGLU) {
              const float g = acc[mi][0][4 * q + e] * rs[mi], u = acc[mi][1][4 * q + e] * rs[mi];
              o[e] = g * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-g * kLog2e)) * u;
            } else {
              o[e] = acc[mi][ti][4 * q + e] * rs[mi];
            }
          }
          *reinterpret_cast<bf16x4*>(wl + l32 * OUT_ROW + (((4 * ti + q) ^ (l32 & 7)) * 16) + 8 * hh) =
              cvt4(o[0], o[1], o[2], o[3]);
        }
#pragma unroll
      for (int k = 0; k < 32 / RPP; ++k) {
        const int rr = lane / CPO + RPP * k, ch = lane % CPO;
        const u32x4 v = *reinterpret_cast<const u32x4*>(wl + rr * OUT_ROW + ((ch ^ (rr & 7)) * 16));
        buf_store16(v, yr, (uint32_t)((int64_t)(brow0 + 32 * mi + rr) * P.ldy * 2) + (uint32_t)(ycol0 * 2 + ch * 16));
      }
    }
    id += step;
    if (id >= t_end) break;
    tile_at(P, id, &mt, &nt);
  }
  waitcnt<0, 15>();   // no stage load left in flight
}

// ---- few rows (M <= 128) ---------------------------------------------------------------
// The product is then a stream of W: a workgroup takes 32 of its rows (SWIGLU: 32 gate rows
// and the 32 up rows of the same columns) and all x rows, its NWV waves taking K blocks of 64 in
// turn; both operands go from global memory straight into MFMA fragments (a W row's 128
// bytes of a block are one line, read by four loads back to back; x stays in L2), and the
// waves' partial products meet in LDS, wave v finishing two (NWV = 8) or four register rows
// of every tile. The row scales come from the x fragments on the way, so the norm needs no
// launch of its own.
// Bound by the stream of W up to 32 rows, by the repeated reads of x from L2 above: K 2048,
// N 11264 (46 MB) with SwiGLU 11.6 us for 1 row and 12.7 for 16 (3.7 TB/s), 18.9 for 64, 29.0 for
// 100 and 29.3 for 128; the 128-row tiles take 36 us for any of them (44 workgroups), which x reads
// would reach past 128 rows.
template <int MB, int NWV>
struct SkinnyGeo {
  static constexpr int TILE = 64 * 16 * 4;       // one wave's partial 32 x 32 tile
  static constexpr int lds(bool swiglu) { return NWV * (swiglu ? 2 : 1) * MB * TILE + NWV * MB * 32 * 4; }
};

template <int MB, int NWV, bool SWIGLU, bool NORM>
__global__ __launch_bounds__(64 * NWV, 1) void proj_skinny_kernel(Params P, float* rstd_out, float eps) {
  constexpr int NB = SWIGLU ? 2 : 1, RW = 16 / NWV;   // W operands; register rows a wave finishes
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int n0 = blockIdx.x * 32, F = P.N >> 1;
  const bf16* wp[NB];
  const bf16* xp[MB];
#pragma unroll
  for (int i = 0; i < NB; ++i) wp[i] = P.w + (int64_t)(n0 + i * F + l32) * P.ldw + 8 * hh;
#pragma unroll
  for (int i = 0; i < MB; ++i) xp[i] = P.x + (int64_t)min(32 * i + l32, P.M - 1) * P.ldx + 8 * hh;

  f32x16 acc[NB][MB];
  float ss[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    ss[m] = 0.f;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][m][r] = 0.f;
  }
  u32x4 wf[2][NB][4], xf[2][MB][4];
  auto load = [&](int set, int b) {
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int s = 0; s < 4; ++s) wf[set][i][s] = *reinterpret_cast<const u32x4*>(wp[i] + 64 * b + 16 * s);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int s = 0; s < 4; ++s) xf[set][i][s] = *reinterpret_cast<const u32x4*>(xp[i] + 64 * b + 16 * s);
  };
  auto mul = [&](int set) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        if (NORM) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float a = bf16lo(xf[set][m][s][e]), b = bf16hi(xf[set][m][s][e]);
            ss[m] += a * a;
            ss[m] += b * b;
          }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i)
          acc[i][m] = mfma32x32x16(__builtin_bit_cast(bf16x8, wf[set][i][s]), __builtin_bit_cast(bf16x8, xf[set][m][s]),
                                   acc[i][m]);
      }
  };
  const int nb = P.K / KT;
  if (w < nb) load(0, w);
  for (int b = w; b < nb; b += 2 * NWV) {
    if (b + NWV < nb) load(1, b + NWV);
    mul(0);
    if (b + NWV < nb) {
      if (b + 2 * NWV < nb) load(0, b + 2 * NWV);
      mul(1);
    }
  }
  // partial tiles: [wave][operand][m][register / 4][lane] of 16 bytes, then the sums of squares
  float* sums = reinterpret_cast<float*>(smem + NWV * NB * MB * SkinnyGeo<MB, NWV>::TILE);
  auto part = [&](int v, int i, int m, int r4) {
    return reinterpret_cast<f32x4*>(smem) + ((((v * NB + i) * MB + m) * 4 + r4) * 64 + lane);
  };
#pragma unroll
  for (int m = 0; m < MB; ++m) {
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        *part(w, i, m, r4) = f32x4{acc[i][m][4 * r4], acc[i][m][4 * r4 + 1], acc[i][m][4 * r4 + 2], acc[i][m][4 * r4 + 3]};
    if (NORM) {
      const float s = halves_sum(ss[m]);
      if (hh == 0) sums[(w * MB + m) * 32 + l32] = s;
    }
  }
  __syncthreads();
  // wave w: registers RW w .. RW w + RW - 1, i.e. columns 8 (r / 4) + 4 hh + r % 4
  const int r0 = RW * w;
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int row = 32 * m + l32;
    float rs = 1.f;
    if (NORM) {
      float s = 0.f;
#pragma unroll
      for (int v = 0; v < NWV; ++v) s += sums[(v * MB + m) * 32 + l32];
      // the caller's scales (P.rstd), or the ones found here
      rs = P.rstd != nullptr ? P.rstd[min(row, P.M - 1)] : __builtin_amdgcn_rsqf(s / (float)P.K + eps);
      if (rstd_out != nullptr && blockIdx.x == 0 && w == 0 && hh == 0 && row < P.M) rstd_out[row] = rs;
    }
    float t[NB][RW];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int e = 0; e < RW; ++e) t[i][e] = 0.f;
#pragma unroll
    for (int v = 0; v < NWV; ++v)
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const float* p = reinterpret_cast<const float*>(part(v, i, m, r0 >> 2)) + (r0 & 3);
#pragma unroll
        for (int e = 0; e < RW; ++e) t[i][e] += p[e];
      }
    float o[RW];
#pragma unroll
    for (int e = 0; e < RW; ++e) {
      if (SWIGLU) {
        const float g = t[0][e] * rs, u = t[NB - 1][e] * rs;
        o[e] = g * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-g * kLog2e)) * u;
      } else {
        o[e] = t[0][e] * rs;
      }
    }
    if (row < P.M) {
      bf16* yp = P.y + (int64_t)row * P.ldy + n0 + 8 * (r0 >> 2) + 4 * hh + (r0 & 3);
      if (RW == 4)
        *reinterpret_cast<bf16x4*>(yp) = cvt4(o[0], o[1], o[RW - 2], o[RW - 1]);
      else
        *reinterpret_cast<uint32_t*>(yp) = __builtin_bit_cast(u32x2, cvt4(o[0], o[1], 0.f, 0.f))[0];
    }
  }
}

}  // namespace mlp
}  // namespace prefixlm
