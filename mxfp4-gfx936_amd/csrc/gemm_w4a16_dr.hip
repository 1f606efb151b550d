// W4A16 routed GEMM with the weights straight into registers (gfx950).
//
// Tile BM x BN (BM = 16 FMX output rows, BN = 64 FN weight rows), 4 waves
// side by side on columns, each wave FN groups of 16 weight rows.  It serves
// expert blocks whose GEMM is bound by the weight stream (up to ~128 routes
// per expert), where the prefill tiles spend their time on 32- to 128-byte
// pieces of weight rows staged through LDS and on a barrier per 64 of K:
//
// * Weights never pass through LDS: per 128-deep unit of K a lane loads 16
//   bytes of its row (a wave instruction covers 64 consecutive bytes of 16
//   rows), a piece of UP units ahead of its use, with no barrier between a
//   wave and its weights.  Bare loads of 201 MB in this pattern read 4.4 TB/s
//   one unit at a time and 5.5-6.1 with both halves of a row's 128-byte lines
//   requested together (UP = 2), which is taken where the registers allow it.
//   On the checkpoint layout a lane's 16 bytes are one 32-value block; four
//   v_permlane swaps per 16 bytes transpose the blocks over the lane groups
//   into the order the prefill tiles multiply in.  The prepacked nibbles
//   (PRE) are in that order already.  Either way the results are bitwise
//   those of the prefill tiles.  They are not those of the 16-row decode
//   kernels, which add K in another order: calls that this kernel takes from
//   them (block_m 16 in dr_faster) differ by rounding, 2e-4 of the 2-norm in
//   bf16, at the same error against 64 bits.
// * The tile's E8M0 bytes (checkpoint layout in both cases) are one
//   contiguous piece of the scale matrix (two with SiLU): copied to LDS once,
//   by 1 KB wave-loads.
// * Activations go global -> LDS in 128-deep stages, two buffers, one barrier
//   per stage (64-deep stages, two barriers: soft op at 509 tokens 64.5 us
//   against 59.2).
// * Row groups of 16 that hold only padding are left out: the tile counts
//   its live groups and runs the loop compiled for that many.
//
// Measured (E=128, top-8, K=2048 N=1536, 3 weight copies rotated, whole soft
// op, prefill tiles -> this): 64 / 128 / 256 / 384 / 509 / 768 tokens 56.7 /
// 57.8 / 60.8 / 67.7 / 76.3 / 80.7 -> 47.4 / 48.9 / 52.1 / 56.5 / 60.0 / 75.5
// us.  With the weight loads left out 32 us of the 509-token GEMM's 52
// remain (decode, LDS reads, MFMAs), without the activation loads 49: the
// stream and the arithmetic of the three resident workgroups still overlap
// only in part.  Deeper weight prefetch (two pieces in flight), 128-column
// tiles on full grids and tile orders that need no routed row count did not
// help.
//
// No spills are allowed here: scratch accesses count in vmcnt out of order
// with the loads, and the stage waits count loads.
#include <algorithm>
#include <cmath>

#include "gemm.h"
#include "silu.h"

namespace mx {
namespace {

template <typename T>
struct V8Of;
template <>
struct V8Of<__bf16> {
  typedef bf16x8 type;
};
template <>
struct V8Of<_Float16> {
  typedef f16x8 type;
};

template <typename T>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  const T x = from_f32<T>(a), y = from_f32<T>(b);
  return (uint32_t)__builtin_bit_cast(uint16_t, x) | ((uint32_t)__builtin_bit_cast(uint16_t, y) << 16);
}

// d[j] of lane group q holds dword j of block q; afterwards d[b] of lane
// group q holds dword q of block b.
__device__ __forceinline__ void transpose_blocks(uint32_t (&d)[4]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const auto s = __builtin_amdgcn_permlane32_swap(d[j], d[j + 2], false, false);
    d[j] = s[0];
    d[j + 2] = s[1];
  }
#pragma unroll
  for (int j = 0; j < 4; j += 2) {
    const auto s = __builtin_amdgcn_permlane16_swap(d[j], d[j + 1], false, false);
    d[j] = s[0];
    d[j + 1] = s[1];
  }
}

struct DrTile {
  int64_t pos0;
  int expert, ncol0, wave, lane;
  uint8_t *sA, *sS;
  int sst;    // LDS bytes of a row's scales
  int spart;  // LDS offset of the up rows' scales (SiLU)
};

template <typename T, int FMX, int FN, int UP, int EPI, bool PRE, int FM>
__device__ __forceinline__ void dr_body(const GemmArgs& g, const DrTile& t) {
  typedef typename V8Of<T>::type V8;
  constexpr int BM = FMX * 16;
  constexpr bool SILU = EPI == EPI_SILU_MUL;
  constexpr int AJ = (FM + 1) / 2;   // wave-loads of 8 rows per wave and stage
  constexpr int A_STAGE = BM * 128;
  const int lane = t.lane, wave = t.wave;
  const int c16 = lane & 15, grp = lane >> 4;

  const i32x4 rA = make_rsrc(g.a, (uint32_t)(g.a_rows * g.lda * (int64_t)sizeof(T)));
  const int64_t b_rows = SILU ? 2 * (int64_t)g.inter : (int64_t)g.n;
  const i32x4 rB = PRE ? make_rsrc(g.pre_b + t.expert * g.pre_b_e,
                                   (uint32_t)prepacked_nibble_bytes(b_rows, g.k))
                       : make_rsrc(g.b + t.expert * g.b_e, (uint32_t)(b_rows * g.b_n));

  uint32_t a_off[AJ];
#pragma unroll
  for (int j = 0; j < AJ; ++j) {
    const int row = (j * 4 + wave) * 8 + (lane >> 3);
    const RowInfo ri = row_info(g, t.pos0 + row);
    a_off[j] = ri.valid ? (uint32_t)(ri.a_row * g.lda * (int64_t)sizeof(T)) +
                              ((lane & 7) ^ (row & 7)) * 16
                        : kOOB;
  }
  uint32_t b_off[FN];
  int s_rd[FN];
#pragma unroll
  for (int fn = 0; fn < FN; ++fn) {
    const int lrow = SILU ? (wave * (FN / 2) + fn / 2) * 16 + c16 : (wave * FN + fn) * 16 + c16;
    const int orow = t.ncol0 + lrow;
    const int64_t grow = (SILU && (fn & 1) ? (int64_t)g.inter : 0) + orow;
    if constexpr (PRE)
      b_off[fn] =
          orow - c16 < g.n ? (uint32_t)((grow >> 4) * (g.k / 64) * 512) + lane * 8 : kOOB;
    else
      b_off[fn] = orow < g.n ? (uint32_t)(grow * g.b_n) + grp * 16 : kOOB;
    s_rd[fn] = (SILU && (fn & 1) ? t.spart : 0) + lrow * t.sst;
  }
  const int nu = g.k / 128;
  // stage u: both 64-deep halves of unit u, in buffer u % 2
  auto issue_a = [&](int u) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < AJ; ++j)
        llvm_amdgcn_raw_buffer_load_lds(
            rA, lds_ptr(t.sA + ((u & 1) * 2 + h) * A_STAGE + (j * 4 + wave) * 1024), 16,
            (int)(u < nu ? a_off[j] : kOOB), u * 256 + h * 128, 0, 0);
  };
  // the piece in flight: per unit and group 16 bytes, one load (checkpoint) or
  // two of the group's 512-byte step blocks (PRE)
  constexpr int WL = PRE ? 2 : 1;
  typedef std::conditional_t<PRE, i32x2, i32x4> WV;
  WV w[UP][FN][WL];
  auto load_w = [&](int p) {
#pragma unroll
    for (int fn = 0; fn < FN; ++fn)
#pragma unroll
      for (int x = 0; x < UP; ++x) {
        const int u = p * UP + x;
        const uint32_t off = u < nu ? b_off[fn] : kOOB;
        if constexpr (PRE) {
          w[x][fn][0] = llvm_amdgcn_raw_buffer_load_v2i32(rB, off, u * 1024, 0);
          w[x][fn][1] = llvm_amdgcn_raw_buffer_load_v2i32(rB, off, u * 1024 + 512, 0);
        } else {
          w[x][fn][0] = llvm_amdgcn_raw_buffer_load_v4i32(rB, off, u * 64, 0);
        }
      }
  };
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  issue_a(0);
  asm volatile("" ::: "memory");
  load_w(0);
  asm volatile("" ::: "memory");

  const int a_rd = c16 * 128 + ((grp ^ (c16 & 7)) * 16);
  const int np = (nu + UP - 1) / UP;
  for (int p = 0; p < np; ++p) {
    uint32_t tw[UP][FN][4];
    static_for<0, UP>([&](auto xx) {
      constexpr int x = decltype(xx)::value;
      const int u = p * UP + x;
      // an odd last unit: nothing past K (its weights read as zero codes, but
      // the scale bytes there are the next row's, and 0 x 255 is NaN)
      if constexpr (x > 0) {
        if (u >= nu) return;
      }
      uint32_t sd[FN];
      // A(u) has landed (only the piece issued after it may be in flight),
      // and this wave's reads of stage u - 1, whose buffer the next loads
      // overwrite, are back
      __builtin_amdgcn_sched_barrier(0);
      wait_vmcnt<(UP == 1 || x == 1) ? UP * FN * WL : 0>();
      wait_lgkm0();
      barrier_only();
      issue_a(u + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
        sd[fn] = *reinterpret_cast<const uint32_t*>(t.sS + s_rd[fn] + u * 4);
      if constexpr (x == 0) {
#pragma unroll
        for (int xi = 0; xi < UP; ++xi)
#pragma unroll
          for (int fn = 0; fn < FN; ++fn) {
            const WV lo = w[xi][fn][0], hi = w[xi][fn][WL - 1];
            const int v2 = PRE ? hi[0] : lo[2 % (PRE ? 2 : 4)];
            const int v3 = PRE ? hi[1] : lo[3 % (PRE ? 2 : 4)];
            uint32_t(&d)[4] = tw[xi][fn];
            // moved out by hand: as plain copies the compiler lets the piece
            // keep these registers, and moves the next piece's over at the
            // loop's end, which waits for its loads
            asm volatile(
                "v_mov_b32 %0, %4\n\tv_mov_b32 %1, %5\n\tv_mov_b32 %2, %6\n\tv_mov_b32 %3, %7"
                : "=&v"(d[0]), "=&v"(d[1]), "=&v"(d[2]), "=&v"(d[3])
                : "v"(lo[0]), "v"(lo[1]), "v"(v2), "v"(v3));
          }
        __builtin_amdgcn_sched_barrier(0);
        load_w(p + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (!PRE) {
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) transpose_blocks(tw[x][fn]);
      }
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const uint8_t* As = t.sA + ((u & 1) * 2 + b / 2) * A_STAGE;
        V8 af[FM], bf[FN];
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
          af[fm] = *reinterpret_cast<const V8*>(As + ((a_rd + fm * 16 * 128) ^ ((b & 1) * 64)));
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
          bf[fn] = Decode<T>::run(tw[x][fn][b], e8m0_scale((sd[fn] >> (8 * b)) & 0xFF));
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
          for (int fm = 0; fm < FM; ++fm) acc[fm][fn] = mfma16(bf[fn], af[fm], acc[fm][fn]);
      }
    });
  }
  wait_vmcnt<0>();  // the direct-to-LDS loads past K, before the LDS is given back

  // ---- epilogue, from the registers: lane owns row fm*16 + c16 and columns
  // fn*16 + grp*4 .. +3 of its wave's piece
  float alpha = scalar_alpha(g, t.expert);
  if constexpr (EPI != EPI_SILU_MUL) {
    if (g.ref_round) {
      ref_pass<std::conditional_t<EPI == EPI_STORE_F32, float, T>>(g, t.expert, acc);
      alpha = 1.0f;
    }
  }
  constexpr int FO = SILU ? FN / 2 : FN;  // output blocks of 16 columns
  const int wcol = t.ncol0 + wave * FO * 16;
#pragma unroll
  for (int fm = 0; fm < FM; ++fm) {
    const RowInfo r = row_info(g, t.pos0 + fm * 16 + c16);
    float rw = 1.0f;
    if (!SILU && g.route_w) rw = r.valid ? g.route_w[r.out_row] : 0.f;
    auto outv = [&](int fo, int i) -> float {
      if constexpr (SILU) {
        // vllm:249-252 on tensors of T: gate and up rounded to T, silu in
        // FP32 rounded to T, the product rounded to T
        const T gb = from_f32<T>(acc[fm][2 * fo][i] * alpha);
        const T ub = from_f32<T>(acc[fm][2 * fo + 1][i] * alpha);
        return to_f32(silu_round<T>(gb)) * to_f32(ub);
      } else {
        // rounded to FP32 before the conversion to T, as in the prefill tiles
        // (the compiler would fold an fp16 conversion into the product)
        float o = acc[fm][fo][i] * alpha * rw;
        if constexpr (std::is_same<T, _Float16>::value) asm("" : "+v"(o));
        return o;
      }
    };
    if constexpr (EPI == EPI_STORE_F32) {
      float* const crow = static_cast<float*>(g.c) + (r.valid ? r.out_row : 0) * g.ldc;
#pragma unroll
      for (int fo = 0; fo < FO; ++fo) {
        const int col = wcol + fo * 16 + grp * 4;
        if (!r.valid || col >= g.n) continue;
        const float o[4] = {outv(fo, 0), outv(fo, 1), outv(fo, 2), outv(fo, 3)};
        if (col + 4 <= g.n && g.ldc % 4 == 0) {
          *reinterpret_cast<f32x4*>(crow + col) = f32x4{o[0], o[1], o[2], o[3]};
        } else {
          for (int i = 0; i < 4 && col + i < g.n; ++i) crow[col + i] = o[i];
        }
      }
    } else {
      T* const crow = static_cast<T*>(g.c) + (r.valid ? r.out_row : 0) * g.ldc;
      constexpr int FP = FO / 2;
#pragma unroll
      for (int fp = 0; fp < FP; ++fp) {
        // lane pairs 16 apart trade halves: each lane then holds 8
        // consecutive columns of one block
        uint32_t pv[2], qv[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          pv[x] = pack2<T>(outv(2 * fp, 2 * x), outv(2 * fp, 2 * x + 1));
          qv[x] = pack2<T>(outv(2 * fp + 1, 2 * x), outv(2 * fp + 1, 2 * x + 1));
          const auto sw = __builtin_amdgcn_permlane16_swap(pv[x], qv[x], false, false);
          pv[x] = sw[0];
          qv[x] = sw[1];
        }
        const int col = wcol + (2 * fp + (grp & 1)) * 16 + (grp & 2) * 4;
        if (!r.valid || col >= g.n) continue;
        const uint32_t v[4] = {pv[0], pv[1], qv[0], qv[1]};
        if (col + 8 <= g.n && g.ldc % 8 == 0) {
          *reinterpret_cast<i32x4*>(crow + col) = i32x4{(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
        } else {
          for (int i = 0; i < 8 && col + i < g.n; ++i)
            crow[col + i] = __builtin_bit_cast(T, (uint16_t)(v[i / 2] >> (16 * (i & 1))));
        }
      }
      if constexpr (FO % 2 == 1) {
        constexpr int fo = FO - 1;
        const int col = wcol + fo * 16 + grp * 4;
        const uint32_t v[2] = {pack2<T>(outv(fo, 0), outv(fo, 1)), pack2<T>(outv(fo, 2), outv(fo, 3))};
        if (r.valid && col < g.n) {
          if (col + 4 <= g.n && g.ldc % 4 == 0) {
            *reinterpret_cast<uint2*>(crow + col) = uint2{v[0], v[1]};
          } else {
            for (int i = 0; i < 4 && col + i < g.n; ++i)
              crow[col + i] = __builtin_bit_cast(T, (uint16_t)(v[i / 2] >> (16 * (i & 1))));
          }
        }
      }
    }
  }
}

template <typename T, int FMX, int FN, int EPI, bool PRE>
__global__ __launch_bounds__(256, FN == 2 ? 4 : 3) void w4a16_dr(GemmArgs g, int nbm, int nbn) {
  constexpr int BM = FMX * 16;
  constexpr int BN = 64 * FN;
  constexpr bool SILU = EPI == EPI_SILU_MUL;
  constexpr int OUT_COLS = SILU ? BN / 2 : BN;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  DrTile t;
  t.lane = threadIdx.x & 63;
  t.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int bm, bn;
  if (!tile_of(g, BM, nbm, nbn, bm, bn, blockIdx.x, gridDim.x)) return;
  t.pos0 = (int64_t)bm * BM;
  t.expert = block_expert(g, t.pos0);
  t.ncol0 = bn * OUT_COLS;
  if (t.expert < 0) {  // aiter:156-172: expert not on this device -> zeros
    for (int idx = threadIdx.x; idx < BM * OUT_COLS; idx += 256) {
      const int r = idx / OUT_COLS, cc = idx % OUT_COLS;
      const RowInfo ri = row_info(g, t.pos0 + r);
      if (ri.valid && t.ncol0 + cc < g.n) {
        if constexpr (EPI == EPI_STORE_F32)
          static_cast<float*>(g.c)[ri.out_row * g.ldc + t.ncol0 + cc] = 0.f;
        else
          static_cast<T*>(g.c)[ri.out_row * g.ldc + t.ncol0 + cc] = from_f32<T>(0.f);
      }
    }
    return;
  }
  t.sA = smem;
  t.sS = smem + BM * 512;
  t.sst = (int)g.bs_n;
  // the tile's scale rows: contiguous, or with SiLU the gate and the up
  // rows (each whole 1 KB pieces: 64 FN / 2 rows of a multiple of 4 bytes)
  {
    const int64_t b_rows = SILU ? 2 * (int64_t)g.inter : (int64_t)g.n;
    const i32x4 rS = make_rsrc(g.bs + t.expert * g.bs_e, (uint32_t)(b_rows * g.bs_n));
    constexpr int PARTS = SILU ? 2 : 1;
    const int part = BN / PARTS * t.sst;  // bytes
    const int per = (part + 1023) / 1024;
    t.spart = per * 1024;
    for (int i = t.wave; i < PARTS * per; i += 4) {
      const int p = i / per, q = i - p * per;
      const int in = q * 1024 + t.lane * 16;
      const uint32_t off = (uint32_t)(((int64_t)p * g.inter + t.ncol0) * g.bs_n) + in;
      llvm_amdgcn_raw_buffer_load_lds(rS, lds_ptr(t.sS + (p * per + q) * 1024), 16,
                                      in < part ? (int)off : (int)kOOB, 0, 0, 0);
    }
    asm volatile("" ::: "memory");
  }
  // live groups of 16 rows: any valid row
  int live = 0;
  {
    const RowInfo ri = row_info(g, t.pos0 + (t.lane < BM ? t.lane : 0));
    const uint64_t m = __ballot(t.lane < BM && ri.valid);
#pragma unroll
    for (int i = 0; i < FMX; ++i)
      if ((m >> (16 * i)) & 0xFFFF) live = i + 1;
  }
  if (live == 0) wait_vmcnt<0>();  // the scale copies, before the LDS is given back
  static_for<1, FMX + 1>([&](auto f) {
    constexpr int FM = decltype(f)::value;
    // two units per piece where the registers of three workgroups per CU
    // (four with FN = 2) hold them; the prepacked blocks are whole lines
    constexpr int UP = (FN == 2 || (!PRE && FM <= 2)) ? 2 : 1;
    if (live == FM) dr_body<T, FMX, FN, UP, EPI, PRE, FM>(g, t);
  });
}

// LDS of a tile: two activation buffers of a 128-deep stage, the scale rows
// (one or two pieces, each rounded up to whole wave-loads).
constexpr int64_t kDrLds = 80 * 1024;  // two workgroups per CU at the longest K
int64_t dr_lds(int bm, int bn, int64_t bs_n) { return bm * 512 + (bn * bs_n + 2047) / 1024 * 1024; }

template <typename T, int FMX, int FN, int EPI, bool PRE>
int launch_dr(const GemmArgs& g, hipStream_t st) {
  constexpr int BM = FMX * 16, BN = 64 * FN;
  const int out_cols = EPI == EPI_SILU_MUL ? BN / 2 : BN;
  const int nbn = (g.n + out_cols - 1) / out_cols;
  const int64_t nbm = (g.m + BM * 8 - 1) / (BM * 8) * 8;  // every XCD covers 1/8 of the capacity (tile_of)
  const int64_t nwg = nbm * nbn;
  if (nwg <= 0 || nwg > 0x7FFFFFFF) {
    set_error("w4a16 routed: bad grid");
    return MXFP4_ERR_VALUE;
  }
  w4a16_dr<T, FMX, FN, EPI, PRE>
      <<<(unsigned)nwg, 256, dr_lds(BM, BN, g.bs_n), st>>>(g, (int)nbm, nbn);
  return launch_status("w4a16 routed launch");
}

template <typename T, int EPI, bool PRE>
int launch_shape(const GemmArgs& g, bool wide, hipStream_t st) {
  if constexpr (!PRE && EPI != EPI_SILU_MUL) {
    if (g.block_m % 64 != 0) {  // a caller's 32-row blocks
      if (wide) return launch_dr<T, 2, 4, EPI, PRE>(g, st);
      return launch_dr<T, 2, 2, EPI, PRE>(g, st);
    }
  }
  if (wide) return launch_dr<T, 4, 4, EPI, PRE>(g, st);
  return launch_dr<T, 4, 2, EPI, PRE>(g, st);
}

template <typename T, int EPI>
int launch_layout(const GemmArgs& g, bool wide, hipStream_t st) {
  if constexpr (EPI != EPI_STORE_F32) {
    if (g.block_m % 64 == 0 && pf_prepacked_usable(g))
      return launch_shape<T, EPI, true>(g, wide, st);
  }
  return launch_shape<T, EPI, false>(g, wide, st);
}

// Expert blocks of `rows` rows that the routes fill when their experts are
// drawn alike: an expert with `avg` routes on average, deviation sqrt(avg),
// has a block beyond j * rows if it has more routes than that.
int64_t dr_blocks(int64_t routes, int64_t experts, int64_t rows) {
  const int64_t busy = std::min(routes, experts);
  if (busy <= 0) return 0;
  const double avg = (double)routes / (double)busy, dev = std::sqrt(avg), r = (double)rows;
  const double sure = std::floor(std::max(0.0, avg - 2.0 * dev) / r);  // P = 1 up to here
  double per = 1.0 + sure;
  for (double over = avg - (sure + 1.0) * r; over > -2.0 * dev; over -= r)
    per += 0.5 + over / (4.0 * dev);
  return (int64_t)((double)busy * per);
}

// 256-column tiles instead of 128-column ones: once there are 1.6 for every
// CU (us of the call on 128-column tiles against 256-column ones, E x K x N at
// routes per expert: 64x2048x1536 at 48, 384 wide tiles, 36.2 against 39.0;
// 32x2048x1536 at 96, 384, 32.5 against 36.6; 64x2048x1536 on 32-row blocks at
// 24, 417, 1.09 times as fast on wide ones; 32x2048x1536 at 128, 480, 45.9
// against 37.5; 64x4096x1024 at 80, 497, 86.7 against 73.0; 128x2048x1536 at
// 16, 768, 57.0 against 52.1).
bool dr_wide(int64_t routes, int64_t experts, int64_t n, bool silu, int rows, int64_t cus) {
  const int out = silu ? 128 : 256;
  return 10 * dr_blocks(routes, experts, rows) * ((n + out - 1) / out) >= 16 * cus;
}

}  // namespace

// Layouts and sizes the kernel takes (routed blocks of a multiple of 32 rows).
bool dr_supported(const GemmArgs& g) {
  if (g.bias) return false;
  if (g.bs_n % 4 != 0 || g.bs_e % 16 != 0 || (reinterpret_cast<uintptr_t>(g.bs) & 15) ||
      g.inter % 16 != 0)
    return false;
  if (dr_lds(64, 128, g.bs_n) > kDrLds) return false;
  return pf_supported(g, 2);
}

// Whether the routed GEMM (n output columns, K = k, `routes` routes over its
// experts) runs faster here, on 64-row blocks (32-row ones of a caller), than
// on the kernels its blocks of `block_m` rows (a caller's, or the ones the
// call would plan without this kernel) take otherwise: the 16-row decode
// kernels, or the prefill tiles.  Figures: us of the whole call in graph
// replays over weights that do not fit the MALL, E x K x N at routes per
// expert, those kernels -> this where it is taken, "vs" where it is not; top-k
// of softmaxed N(0, 1) logits, "skewed" with an N(0, 1) bias per expert.
bool dr_faster(int64_t routes, int64_t experts, int64_t n, int64_t k, bool silu, bool prepacked,
               int block_m, int64_t cus) {
  const double avg = (double)routes / (double)experts;
  const int64_t busy = std::min(routes, experts);
  const int64_t wide = (n + (silu ? 127 : 255)) / (silu ? 128 : 256);  // column tiles
  const int64_t narrow = (n + (silu ? 63 : 127)) / (silu ? 64 : 128);
  // a grid of less than two 256-column tiles per CU when every expert has
  // one block
  const bool small = busy * wide < 2 * cus;
  // 128-row blocks leave half of the CUs idle (long K only)
  const bool idle = k >= 2048 && 2 * dr_blocks(routes, experts, 128) * wide <= cus;
  if (!prepacked) {
    if (avg <= 1.5) return false;
    if (block_m == 16) {
      // Against the decode kernels, whose waves split K: not on grids of
      // less than two 128-column tiles per CU (soft op, 32x2048x1536 at 3 / 4
      // 21.8 / 22.9 vs 23.9 / 24.0, skewed 16.4 / 19.2 vs 21.1 / 22.2; layer,
      // 32x2048x768 at 3 / 6 34.0 / 35.9 vs 36.7 / 37.4), and from 2.5 routes
      // per expert unless the experts cover half of the CUs (soft op,
      // 64x4096x1024 at 2 / 3 37.5 vs 38.9 / 43.0 -> 40.2; layer,
      // 64x1024x1408 at 2 44.3 vs 45.8; 64x1024x512 26.3 -> 24.5 and
      // 64x2048x1024 57.5 -> 55.0 at 2 are given up; 128x2048x768 at 2 / 3
      // 79.8 / 86.3 -> 76.4 / 80.5)
      return busy * narrow >= 2 * cus && (avg > 2.5 || 2 * busy >= cus);
    }
    if (block_m % 128 == 0) {
      // Against 128-row tiles: on small grids up to 128 routes per expert
      // (32x2048x1536 at 96 / 128 41.2 / 54.8 -> 32.7 / 47.9) and while even
      // those tiles leave CUs idle (16x2048x1536 at 192 40.0 -> 30.8); on
      // full grids less the shorter K is (64x768x2048 at 48 / 64 28.6 -> 27.7
      // / 29.1 vs 30.9; 128x2048x1536 at 48 / 80 87.8 -> 82.3 / 93.4 vs 95.3;
      // 128x4096x1024 at 80 / 96 143.3 -> 132.3 / 146.6 vs 145.1)
      if (small) return avg <= 128.0 || dr_blocks(routes, experts, 128) * wide < cus;
      return avg <= (k >= 4096 ? 80.0 : (k >= 2048 ? 64.0 : 48.0));
    }
    if (block_m % 64 != 0 && k < 2048) {
      // 32-row tiles, short K: 64x768x2048 at 20 / 32 / 48 21.4 / 24.5 ->
      // 17.7 / 21.6 / 28.6 vs 29.4; 8x768x2048 at 64 / 128 9.8 -> 9.1 / 11.4
      // vs 11.6
      return avg <= (busy * wide < cus ? 64.0 : 32.0);
    }
    if (block_m % 64 == 0 && !dr_wide(routes, experts, n, silu, 64, cus) && avg > 96.0) {
      // 64-row tiles of the same grid, many rows: only where CUs idle
      // (8x4096x1024 at 128 41.5 -> 31.2; 8x768x2048 at 96 / 128 11.1 -> 10.8
      // / 12.1 vs 13.4; 16x2048x1536 at 192 30.3 vs 31.3)
      return idle;
    }
    // full grids of long K up to 80 (128x2048x1536 at 64 / 80 / 96 1.10 / 1.15
    // / 1.14 times as fast on a caller's 64-row blocks, 1.00 / 1.06 / 1.05 on
    // 32-row ones; 64x2048x1536, 32-row, at 96 68.2 vs 68.6)
    return avg <= ((small || k < 2048) ? 128.0 : 80.0) || idle;
  }
  // Prepacked (MoE layer).  Against the 16-row decode kernels at <= 1.5 routes
  // per expert: 16 / 24 tokens of 128x2048x768 63.5 / 74.5 -> 58.1 / 69.3.
  if (avg <= 1.5) return true;
  // Grids of less than 1.5 64-column tiles per CU: 16x2048x768 at 6 / 16 / 32
  // / 64 / 96 33.9 / 34.4 / 35.4 / 52.4 / 53.2 -> 28.4 / 29.2 / 32.0 / 46.1 /
  // 46.8.
  if (2 * busy * narrow < 3 * cus) return avg > 2.0 && avg <= 96.0;
  // Others: the 32-row tiles, whose grid is one round, up to ~28 routes per
  // expert on small ones (32x2048x768 at 8 / 16 / 28 35.9 / 37.1 / 39.8 vs
  // 35.0 / 36.5 / 40.5, skewed 36.4 / 38.1 / 42.2 vs 44.8 / 45.4 / 47.6; at 32
  // 44.5 -> 41.4, skewed 43.0 -> 47.1), then this up to 64 where its tiles are
  // at most one per CU (32x2048x768 at 48 / 64 / 96 54.7 / 58.4 -> 49.3 / 58.1
  // / 61.7 vs 62.4; 64x2048x768, with 1.5, 79.2 vs 87.6 at 64); K >= 4096 at 4
  // / 8 59.8 / 60.5 -> 56.2 / 57.6 (32x4096x1024).  On full ones this from 20
  // to 32 (128x2048x768 at 20 / 24 / 32 / 40 82.4 vs 86.3 / 95.4 / 94.9 ->
  // 87.2 / 94.1 / 102.7 vs 107.3; 128x4096x1024 at 24 / 32 224.6 / 240.9 ->
  // 198.6 / 210.9).  Skewed routing turns 24 to 32 round on short K
  // (128x2048x768 84.1 / 111.7 -> 94.3 / 116.9; 128x4096x1024 0.96 / 1.00 of
  // the rate): the host does not know the counts.
  if (small) {
    if (busy * wide <= cus && ((avg > 28.0 && avg <= 64.0) || (k >= 4096 && avg > 2.0 && avg <= 8.0)))
      return true;
    return avg > 28.0 && avg <= 32.0;
  }
  return avg > 20.0 && avg <= 32.0;
}

int launch_w4a16_dr(const GemmArgs& g, int dtype, int epi, hipStream_t st) {
  const int bm = g.block_m % 64 == 0 ? 64 : 32;
  const bool wide = dr_wide(g.num_valid, g.num_experts, g.n, epi == EPI_SILU_MUL, bm,
                            device_cus()) &&
                    dr_lds(bm, 256, g.bs_n) <= kDrLds;
  if (dtype == MXFP4_DT_BF16) {
    switch (epi) {
      case EPI_STORE: return launch_layout<__bf16, EPI_STORE>(g, wide, st);
      case EPI_STORE_F32: return launch_layout<__bf16, EPI_STORE_F32>(g, wide, st);
      default: return launch_layout<__bf16, EPI_SILU_MUL>(g, wide, st);
    }
  }
  if (epi == EPI_STORE_F32) {
    set_error("w4a16 routed: C in FP32 takes bf16 activations only");
    return MXFP4_ERR_TYPE;
  }
  return epi == EPI_STORE ? launch_layout<_Float16, EPI_STORE>(g, wide, st)
                          : launch_layout<_Float16, EPI_SILU_MUL>(g, wide, st);
}

}  // namespace mx

// For the tests (not in the public header): columns of the tile a routed GEMM
// on blocks of block_m rows gets on a chip of `cus` CUs, 0 where it stays on
// the other kernels.  rows: of this kernel's tiles, 32 or 64.
extern "C" int mxfp4_test_dr_columns(int64_t routes, int64_t experts, int64_t n, int64_t k,
                                     int silu, int prepacked, int block_m, int rows, int64_t cus) {
  using namespace mx;
  if (!dr_faster(routes, experts, n, k, silu, prepacked, block_m, cus) ||
      dr_lds(64, 128, k / 32) > kDrLds)
    return 0;
  return dr_wide(routes, experts, n, silu, rows, cus) && dr_lds(rows, 256, k / 32) <= kDrLds ? 256
                                                                                            : 128;
}
