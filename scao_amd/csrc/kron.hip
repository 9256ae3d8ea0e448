// Kronecker-block kernels of the SCAO step on gfx950 (fp32 MFMA 16x16x4).
//
// Per block (m x n, rank k) the reference computes, in
// scao/cuda/__init__.py:78-99 (the path scao/preconditioner.py:519 takes):
//     P = (U_l^T G) U_r ;  Delta = (s_l s_r^T - 1) * P ;  out = G + (U_l Delta) U_r^T
// and, for the curvature clip (scao/preconditioner.py:558-564), the Frobenius
// norm of clamp(S_l,eps)^-1/2 * P * clamp(S_r,eps)^-1/2.  Here that is four
// kernels so every block of every parameter runs in one launch per stage:
//   project  T = U_l^T G                 (4mnk/2 flops, reads G once; MFMA)
//   delta    P = T U_r, Delta, nu^2      (k x k per block)
//   lift     W = U_l Delta               (m x k per block)
//   apply    out = G + W U_r^T, fused with the optimizer's elementwise tail
//
// Lane layouts.  For v_mfma_f32_16x16x4_f32 lane l supplies A[l%16][l/16],
// B[l/16][l%16] and receives D[4*(l/16)+r][l%16].  Two index permutations keep
// global accesses vectorised:
//   * output columns: MFMA tile t, column jj maps to matrix column
//     j0 + 4*jj + t, so one float4 per lane feeds (or receives) four tiles;
//   * reduction index: K-step s of a 16-wide chunk uses index
//     kb + 4*(l/16) + s, so one float4 per lane feeds four K-steps.
// Both only reorder an exact sum, so they change rounding order, never terms.
#include <algorithm>
#include <mutex>

#include "scao_common.hpp"

using namespace scao;

namespace {

// ----------------------------------------------------------- project ---
// T[c0:c0+CR, j0:j0+256] = U_l^T G over rows [i_beg, i_end), on the bf16
// matrix cores with fp32 products through three-way splits (mfma_x6).  Rows
// are consumed in chunks of PR = 32, one v_mfma_f32_16x16x32 deep.  NT
// threads (NT / 64 waves) share the CR x 256 tile; wave w owns
// CW = 256 / (NT / 64) columns (NJ = CW / 16 output tiles across) and all CR
// rows of T.
//   * G does not pass through LDS: lane (jj, g) of wave w loads rows
//     8g..8g+7 of the chunk at the NJ columns j0 + CW*w + NJ*jj + t, which is
//     exactly its B operand of the NJ output tiles t (the column permutation
//     of the fp32 form), and splits it in registers.  bf16 gradients are
//     their own split (the two remainders are zero), so their products take
//     three MFMAs instead of six and no split.
//   * U_l (shared by the waves) is split by its loader and stored as three
//     bf16 planes, column-major inside the chunk (column pitch 80 B: the 16
//     lanes of one A-operand read hit 16 disjoint bank quads).
// The next chunk's G, p and U_l are loaded while the current one's MFMAs run.
// Chunk-0 tasks also reduce ||g||^2 and ||p*decay||^2 of their rows and strip
// from the loaded registers (every element passes through exactly one lane).
//
// EDGE: the strip may end past column n and the rows past i_end (those count
// as zero); every load is masked and G has type DT.
// KEDGE: c0 + CR may lie past k, so U_l's loads and T's stores are masked.
// Loads need element alignment only, in every form.
//
// When the whole tiles of a step are too few to fill 256 CUs the rows are
// split (SCAO_LF_NSPLIT_SHIFT): each part writes a plane of its own and the
// delta stage adds the planes in order.
//
// HBM bounds the projection of a step that fills the chip (5.4 TB/s at 323 M
// parameters, k = 64), latency a smaller one.  Against fp32 MFMAs over tiles
// staged through LDS with masked scalar loads, for all but aligned whole fp32
// tiles: one Llama-1B layer in bf16 866 -> 75 us, odd sizes (7 M elements) 596
// -> 66 us; row parts: one GPT-2-small layer 80 -> 19 us.
constexpr int PR = 32;           // rows per chunk
// a lane's rows are addressed by 32-bit byte offsets: 24 row strides and a
// strip stay below 2^32 for strides under 2^25 elements
constexpr int64_t SHORT_ROWS = 1 << 25;

// rows of one part of a block's row split, and the part's plane of T: plane
// 0 (T itself) when the rows are whole, else plane 1 + part
__host__ __device__ inline int split_rows(int m, int parts) {
  return ((m + PR * parts - 1) / (PR * parts)) * PR;
}
__host__ __device__ inline int64_t plane_floats(int64_t n) { return (n + 3) & ~(int64_t)3; }

// The values one lane holds of a chunk of G or p: eight rows of NJ columns,
// as loaded (DT = SCAO_F32: floats, also in EDGE tiles of any type;
// SCAO_BF16 / SCAO_F16: packed 16-bit pairs).
template <int DT, int NJ> struct lane_rows {
  static constexpr int W = DT == SCAO_F32 ? NJ : NJ / 2;   // 32-bit words per row
  typedef uint32_t vw __attribute__((ext_vector_type(W)));
  typedef vw vwu __attribute__((aligned(DT == SCAO_F32 ? 4 : 2)));
  typedef __attribute__((address_space(1))) vwu gvw;
  vw x[8];
  __device__ __forceinline__ void load(int e, const char* at) {
    x[e] = __builtin_nontemporal_load((const gvw*)at);
  }
  __device__ __forceinline__ float get(int e, int t) const {
    if constexpr (DT == SCAO_F32) return __uint_as_float(x[e][t]);
    const uint32_t u = x[e][t / 2];
    if constexpr (DT == SCAO_BF16) return __uint_as_float(t & 1 ? u & 0xffff0000u : u << 16);
    return f16_to_f((uint16_t)(t & 1 ? u >> 16 : u));
  }
  // column t's bf16 values of all eight rows, as the MFMA takes them
  __device__ __forceinline__ v8bf column(int t) const {
    v4u_t r;
#pragma unroll
    for (int p = 0; p < 4; ++p)
      r[p] = __builtin_amdgcn_perm(x[2 * p + 1][t / 2], x[2 * p][t / 2],
                                   t & 1 ? 0x07060302u : 0x05040100u);
    return __builtin_bit_cast(v8bf, r);
  }
};

constexpr int UCP = 40;   // bf16 per U_l column in LDS (32 rows + pad)
template <int CR> struct project_lds {
  __bf16 U[2][3][CR][UCP];   // by chunk parity
  double red[16];
};

template <bool DO_P, int CR, int NT, int DT, bool EDGE, bool KEDGE = EDGE>
__device__ __forceinline__ void project_tile(project_lds<CR>& lds, const scao_leaf_desc& L, const scao_param_desc& P,
                                             int j0, int c0, int i_beg, int i_end, float* T,
                                             int slot, double* slots) {
  static_assert(CR == 64 || CR == 128 || CR == 256, "CR");
  static_assert(NT == 256 || NT == 512, "NT");
  static_assert(!EDGE || (DT == SCAO_F32 && (KEDGE || CR == 64)), "EDGE tiles convert on load");
  constexpr int NQ = CR / 16;        // MFMA tiles down T
  constexpr int CW = 256 / (NT / 64);
  constexpr int NJ = CW / 16;        // MFMA tiles across, G columns per lane
  constexpr int UG = NT / 8;         // U_l loader threads per 4-row group
  constexpr int UW = CR / UG;        // U_l columns per loader thread
  constexpr int ES = DT == SCAO_F32 ? 4 : 2;   // bytes per element (EDGE: not used)
  static_assert(UW == 2 || UW == 4, "U_l loader width");
  __bf16 (*Us)[3][CR][UCP] = lds.U;
  const int tid = threadIdx.x;
  const int w = tid / 64, l = tid % 64;
  const int jj = l % 16, g = l / 16;
  const int n = L.n, k = L.k;
  const int64_t ld = L.ld;
  const int dt = EDGE ? P.dtype : DT;
  const bool do_norms = (c0 == 0) && slot >= 0;
  // x * 1.0f == x bit for bit, so no per-element select on the decay flag
  const float dec = (P.flags & SCAO_PF_DECAY) ? P.decay : 1.0f;
  const int gcol = j0 + CW * w + NJ * jj;
  // U_l loader: rows 4*ua .. 4*ua+3 of the chunk, columns ub*UW .. +UW-1
  const int ua = tid / UG, ub = tid % UG;
  // Every load address is a row origin shared by the block (scalar
  // registers) plus a 32-bit lane offset fixed for the whole tile: lane
  // (jj, g) reads rows 8g.. of the chunk at column gcol, the U_l loader rows
  // 4ua.. at column c0 + ub*UW.
  const uint32_t g_lane = (uint32_t)((8 * g * ld + (gcol - j0)) * (int64_t)ES);
  const uint32_t u_lane = (uint32_t)((4 * ua * (int64_t)k + ub * UW) * (int64_t)sizeof(float));
  const int64_t ldb = ld * (int64_t)ES, kb = k * (int64_t)sizeof(float);

  v4f acc[NQ][NJ];
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int t = 0; t < NJ; ++t) acc[q][t] = v4f{0.f, 0.f, 0.f, 0.f};
  double g2 = 0.0, p2 = 0.0;

  lane_rows<DT, NJ> rg, rp;
  float ru[4][UW];
  // Masked rows: every address is clamped into the tile and what lies outside
  // becomes zero afterwards, so the loads of a chunk go out together.
  auto load_edge = [&](lane_rows<DT, NJ>& r, const void* base, int i0) {
    if constexpr (EDGE) {
      const int64_t first = L.off + gcol;
      auto row = [&](int e) { return (int64_t)min(i0 + 8 * g + e, i_end - 1) * ld; };
      if (gcol + NJ <= n && dt == SCAO_F32) {
#pragma unroll
        for (int e = 0; e < 8; ++e) r.load(e, (const char*)((const float*)base + first + row(e)));
      } else if (gcol + NJ <= n) {
        v2u h[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = gld2w((const uint16_t*)base + first + row(e));
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int t = 0; t < NJ; ++t) {
            const uint16_t x = (uint16_t)(t & 1 ? h[e][t / 2] >> 16 : h[e][t / 2]);
            r.x[e][t] = __float_as_uint(dt == SCAO_BF16 ? bf16_to_f(x) : f16_to_f(x));
          }
      } else {
        int64_t col[NJ];
#pragma unroll
        for (int t = 0; t < NJ; ++t) col[t] = L.off + min(gcol + t, n - 1);
        if (dt == SCAO_F32) {
#pragma unroll
          for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int t = 0; t < NJ; ++t) r.x[e][t] = gld1((const uint32_t*)base + col[t] + row(e));
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int t = 0; t < NJ; ++t) r.x[e][t] = ((const gu16*)base)[col[t] + row(e)];
#pragma unroll
          for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int t = 0; t < NJ; ++t) {
              const uint16_t x = (uint16_t)r.x[e][t];
              r.x[e][t] = __float_as_uint(dt == SCAO_BF16 ? bf16_to_f(x) : f16_to_f(x));
            }
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int t = 0; t < NJ; ++t)
          if (i0 + 8 * g + e >= i_end || gcol + t >= n) r.x[e][t] = 0u;
    }
  };
  auto load_g = [&](int i0) {
    if constexpr (EDGE) {
      load_edge(rg, P.graw, i0);
      if (DO_P) load_edge(rp, P.p, i0);
    } else {
      const int64_t o = (L.off + (int64_t)i0 * ld + j0) * ES;
      const char* gb = (const char*)P.graw + o;
      const char* pb = (const char*)P.p + o;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        rg.load(e, gb + e * ldb + g_lane);
        if (DO_P) rp.load(e, pb + e * ldb + g_lane);
      }
    }
  };
  auto load_u = [&](int i0) {
    if constexpr (EDGE || KEDGE) {
      const int col = c0 + ub * UW;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float* src = L.Ul + (int64_t)min(i0 + 4 * ua + r, i_end - 1) * k;
#pragma unroll
        for (int c = 0; c < UW; ++c) ru[r][c] = gld1(src + (KEDGE ? min(col + c, k - 1) : col + c));
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < UW; ++c)
          if (i0 + 4 * ua + r >= i_end || (KEDGE && col + c >= k)) ru[r][c] = 0.f;
    } else {
      const char* ubase = (const char*)(L.Ul + (int64_t)i0 * k + c0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float* src = (const float*)(ubase + r * kb + u_lane);
        if constexpr (UW == 4) {
          const v4f x = gld4(src);
#pragma unroll
          for (int c = 0; c < 4; ++c) ru[r][c] = x[c];
        } else {
          const v2u x = gld2w(src);
          ru[r][0] = __uint_as_float(x[0]);
          ru[r][1] = __uint_as_float(x[1]);
        }
      }
    }
  };

  // U_l's planes for chunk i sit in Us[i & 1]: chunk i+1's are split and
  // written during chunk i (its raw rows were loaded a chunk earlier), so one
  // barrier per chunk separates a buffer's readers from its next writers
  auto write_u = [&](int buf) {
#pragma unroll
    for (int c = 0; c < UW; ++c) {
      // four rows of one column: one 8-byte write per plane
      v2u pl[3];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t a, b, cc;
        split3_pk(ru[2 * h][c], ru[2 * h + 1][c], a, b, cc);   // rows 2h (low), 2h+1
        pl[0][h] = a;
        pl[1][h] = b;
        pl[2][h] = cc;
      }
      const int col = ub * UW + c;
#pragma unroll
      for (int pp = 0; pp < 3; ++pp) *(v2u*)&Us[buf][pp][col][4 * ua] = pl[pp];
    }
  };
  // CR = 256: the prefetches are unconditional, clamped to the last chunk
  // ((i_end - i_beg) % PR == 0 for these tiles), and pinned ahead of the
  // MFMAs: behind a branch, the join makes the compiler wait for every load in
  // flight, the next chunk's G included, and the scheduler sinks them among
  // the MFMAs.  The narrower tiles have half or a quarter of the MFMAs per
  // chunk to hide loads behind and measured faster with the branch (the last
  // chunk loads nothing).
  constexpr bool PIN = CR == 256 && !EDGE && !KEDGE;
  const int last = i_end - PR;
  load_g(i_beg);
  load_u(i_beg);
  write_u(0);
  if (PIN || i_beg + PR < i_end) load_u(PIN && i_beg + PR > last ? last : i_beg + PR);
  __syncthreads();
  for (int i0 = i_beg, cur = 0; i0 < i_end; i0 += PR, cur ^= 1) {
    // this chunk's G operands, split in registers
    bf3 bg[NJ];
#pragma unroll
    for (int t = 0; t < NJ; ++t) {
      if constexpr (DT == SCAO_BF16) {
        bg[t].h = rg.column(t);
      } else {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = rg.get(e, t);
        bg[t] = split_bf3(x);
      }
    }
    if (do_norms) {
      float a = 0.f, b = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int t = 0; t < NJ; ++t) {
          const float y = rg.get(e, t);
          a = fmaf(y, y, a);
          if (DO_P) {
            float x = rp.get(e, t) * dec;
            if (EDGE || DT != SCAO_F32) x = round_to(dt, x);
            b = fmaf(x, x, b);
          }
        }
      g2 += (double)a;
      p2 += (double)b;
    }
    if constexpr (PIN) {
      write_u(cur ^ 1);                   // chunk i+1's planes, read after the barrier below
      // the loads go out after the split (measured faster than letting the
      // scheduler hoist them above it)
      __builtin_amdgcn_sched_barrier(0);
      load_g(i0 + PR < last ? i0 + PR : last);   // in flight during the MFMAs below
      load_u(i0 + 2 * PR < last ? i0 + 2 * PR : last);
      __builtin_amdgcn_sched_barrier(0);
    } else if (i0 + PR < i_end) {
      write_u(cur ^ 1);
      load_g(i0 + PR);
      if (i0 + 2 * PR < i_end) load_u(i0 + 2 * PR);
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      bf3 au;
      au.h = *(const v8bf*)&Us[cur][0][16 * q + jj][8 * g];
      au.m = *(const v8bf*)&Us[cur][1][16 * q + jj][8 * g];
      au.l = *(const v8bf*)&Us[cur][2][16 * q + jj][8 * g];
#pragma unroll
      for (int t = 0; t < NJ; ++t)
        acc[q][t] = DT == SCAO_BF16 ? mfma_x3(au, bg[t].h, acc[q][t])
                                    : mfma_x6(au, bg[t], acc[q][t]);
    }
    __syncthreads();
  }
  // T[c][j] for c = c0 + 16q + 4g + r, j = gcol + t
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int c = c0 + 16 * q + 4 * g + r;
      if constexpr (EDGE || KEDGE) {
        if (c >= k) continue;
#pragma unroll
        for (int t = 0; t < NJ; ++t)
          if (gcol + t < n) gst1(T + (int64_t)c * n + gcol + t, acc[q][t][r]);
      } else {
        typedef float vj __attribute__((ext_vector_type(NJ)));
        typedef vj vju __attribute__((aligned(4)));
        vj o;
#pragma unroll
        for (int t = 0; t < NJ; ++t) o[t] = acc[q][t][r];
        *(__attribute__((address_space(1))) vju*)(T + (int64_t)c * n + gcol) = o;
      }
    }
  if (do_norms) {
    double x[2] = {g2, p2};
    block_sum_n<2, NT>(x, lds.red);
    if (threadIdx.x == 0) {
      slots[(int64_t)slot * SCAO_SLOT_WIDTH + 0] = x[0];
      slots[(int64_t)slot * SCAO_SLOT_WIDTH + 1] = x[1];
      slots[(int64_t)slot * SCAO_SLOT_WIDTH + 2] = 0.0;
    }
  }
}

// A task's part of the row split (a step's ranks are whole multiples of 64, so
// T's rows are): tk.b holds the column origin c0 in its low
// 16 bits and the part above them.
template <bool DO_P, int CR, int NT, int DT, bool EDGE>
__device__ __forceinline__ void project_part(project_lds<CR>& lds, const scao_leaf_desc& L, const scao_param_desc& P,
                                             int j0, int b, int slot, double* slots) {
  const int parts = SCAO_LF_GET_NSPLIT(L.flags), part = b >> 16;
  const int rows = split_rows(L.m, parts);
  const int i_beg = part * rows, i_end = min(L.m, i_beg + rows);
  float* T = L.T + (parts > 1 ? (1 + part) * plane_floats((int64_t)L.k * L.n) : 0);
  project_tile<DO_P, CR, NT, DT, EDGE, false>(lds, L, P, j0, b & 0xffff, i_beg, i_end, T, slot, slots);
}

// ------------------------------------------------------------- delta ---
// P[c0:c0+64, d0:d0+64] = T U_r; Delta and the natural-norm partial.
// The four waves split the n-reduction (one quarter each, 16-column chunks,
// one chunk prefetched); every wave accumulates the whole 64x64 tile
// (16 MFMA tiles) and the four partial tiles are added in LDS in a fixed
// order.  P column d of tile t sits at lane column jj with d = d0 + 4*jj + t,
// so one float4 of a U_r row feeds all four tiles.
constexpr int DP = 64 + 4;   // LDS pitch of a partial tile

// acc[q][t] += sum over j in [jbeg, jend) of A[r0 + 16q + i][j] * B[j][c0 + 4i + t]
// (i = lane % 16) for a 64 x 64 output tile, with the products on the bf16
// matrix cores: six per fp32 product over three-way splits, as the
// projection.  The reduction runs in chunks of 32: lane (i, g) takes A row
// r0 + 16q + i at columns j + 8g .. j + 8g + 7 (the A operand of row tile q)
// and B rows j + 8g .. j + 8g + 7 at columns c0 + 4i .. c0 + 4i + 3 (element t
// of each float4 is the B operand of column tile t), so the accumulator layout
// is the fp32 16x16x4 form's with the same column permutation.  Rows of A and
// B are 16-byte aligned and jend - jbeg is a multiple of 32.
__device__ __forceinline__ void mm64_x6(const float* __restrict__ A, int64_t lda,
                                        const float* __restrict__ B, int64_t ldb, int r0, int c0,
                                        int jbeg, int jend, v4f (&acc)[4][4]) {
  const int l = threadIdx.x % 64, i = l % 16, g = l / 16;
  // each operand's next-chunk load goes out as soon as its current value is
  // split, into the same registers; on the last chunk the loads repeat it
  // (in bounds, unused), so no branch makes the compiler wait for them
  v4f ca[4][2], cb[8];
  auto load_a = [&](int jb, int q, v4f (&a)[2]) {
    const float* ap = A + (int64_t)(r0 + 16 * q + i) * lda + jb + 8 * g;
    a[0] = gld4(ap);
    a[1] = gld4(ap + 4);
  };
  auto load_b = [&](int jb, v4f (&b)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) b[e] = gld4(B + (int64_t)(jb + 8 * g + e) * ldb + c0 + 4 * i);
  };
  if (jbeg >= jend) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) load_a(jbeg, q, ca[q]);
  load_b(jbeg, cb);
  for (int jb = jbeg; jb < jend; jb += 32) {
    const int jn = jb + 32 < jend ? jb + 32 : jb;
    bf3 bt[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = cb[e][t];
      bt[t] = split_bf3(x);
    }
    load_b(jn, cb);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = ca[q][0][e];
        x[4 + e] = ca[q][1][e];
      }
      const bf3 aq = split_bf3(x);
      load_a(jn, q, ca[q]);
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[q][t] = mfma_x6(aq, bt[t], acc[q][t]);
    }
  }
}

// Ps (three partial tiles) and red live in the caller's LDS, so a kernel
// holding both instantiations allocates them once.
template <bool FAST, bool X6 = false>
__device__ __forceinline__ void delta_tile(const scao_leaf_desc& L, float eps, int c0, int d0,
                                           int slot, double* slots, float (*Ps)[64][DP],
                                           double* red) {
  static_assert(FAST || !X6, "X6 needs whole tiles");
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  const int n = L.n, k = L.k;
  const int kk = l / 16;
  const float* T = L.T;
  const float* Ur = L.Ur;
  const int dl = d0 + 4 * (l % 16);      // this lane's 4 P columns
  int dmask = 15;
  if (!FAST)
    for (int t = 0; t < 4; ++t) dmask = (dl + t < k) ? dmask : (dmask & ~(1 << t));
  const bool uvec = FAST || dmask == 15;
  const int nq = ((n + 63) / 64) * 16;    // per-wave share of n, multiple of 16
  const int jbeg = w * nq, jend = min(n, jbeg + nq);

  v4f acc[4][4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[q][t] = v4f{0.f, 0.f, 0.f, 0.f};

  if constexpr (X6) {
    // whole tiles, n % 128 == 0: each wave's quarter of n is a multiple of 32
    mm64_x6(T, n, Ur, k, c0, d0, jbeg, jend, acc);
  } else {
    v4f ra[4], rb[4], na[4], nb[4];
    auto load = [&](int jb, v4f (&a)[4], v4f (&b)[4]) {
      const int j = jb + 4 * kk;
      int jm = 15;
      if (!FAST)
        for (int s2 = 0; s2 < 4; ++s2) jm = (j + s2 < jend) ? jm : (jm & ~(1 << s2));
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = c0 + 16 * q + (l % 16);
        if (FAST)
          a[q] = gld4(T + (int64_t)c * n + j);
        else
          a[q] = (c < k && jm) ? ldf4(T, (int64_t)c * n + j, jm == 15, jm)
                               : v4f{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2) {
        if (FAST)
          b[s2] = gld4(Ur + (int64_t)(j + s2) * k + dl);
        else
          b[s2] = (((jm >> s2) & 1) && dmask) ? ldf4(Ur, (int64_t)(j + s2) * k + dl, uvec, dmask)
                                              : v4f{0.f, 0.f, 0.f, 0.f};
      }
    };
    if (jbeg < jend) load(jbeg, ra, rb);
    for (int jb = jbeg; jb < jend; jb += 16) {
      if (jb + 16 < jend) load(jb + 16, na, nb);
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int t = 0; t < 4; ++t) acc[q][t] = mfma16(ra[q][s2], rb[s2][t], acc[q][t]);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        ra[q] = na[q];
        rb[q] = nb[q];
      }
    }
  }
  // partial tiles of waves 1..3 go through LDS; wave 0 adds them in order
  // (((w0 + w1) + w2) + w3) and finishes its 64 elements per lane:
  // element (16q + 4*kk + r, 4*(l%16) + t)
  if (w > 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *(v4f*)&Ps[w - 1][16 * q + 4 * kk + r][4 * (l % 16)] =
            v4f{acc[q][0][r], acc[q][1][r], acc[q][2][r], acc[q][3][r]};
  }
  __syncthreads();
  const bool sinv4 = L.flags & SCAO_LF_SINV4;
  double nu2 = 0.0;
  if (w == 0) {
    float sr4[4], ir2[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int d = dl + t;
      const float sr = d < k ? gld1(L.Sr + d) : 1.f;
      sr4[t] = sinv4 ? sr : inv4(sr);
      ir2[t] = sinv4 ? 0.f : inv2(sr, eps);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * q + 4 * kk + r;
        const int c = c0 + row;
        if (c >= k) continue;
        const float sl = gld1(L.Sl + c);
        const float sl4 = sinv4 ? sl : inv4(sl);
        const float il2 = sinv4 ? 0.f : inv2(sl, eps);
        const v4f p1 = *(const v4f*)&Ps[0][row][4 * (l % 16)];
        const v4f p2 = *(const v4f*)&Ps[1][row][4 * (l % 16)];
        const v4f p3 = *(const v4f*)&Ps[2][row][4 * (l % 16)];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int d = dl + t;
          if (d >= k) continue;
          const float pv = ((acc[q][t][r] + p1[t]) + p2[t]) + p3[t];
          gst1(L.Delta + (int64_t)c * k + d, (sl4 * sr4[t] - 1.0f) * pv);
          if (!sinv4) {
            const float y = (il2 * pv) * ir2[t];
            nu2 += (double)y * (double)y;
          }
        }
      }
  }
  if (slot >= 0) {
    double xs[1] = {nu2};
    block_sum<1>(xs, red);
    if (threadIdx.x == 0) {
      slots[(int64_t)slot * SCAO_SLOT_WIDTH + 0] = 0.0;
      slots[(int64_t)slot * SCAO_SLOT_WIDTH + 1] = 0.0;
      slots[(int64_t)slot * SCAO_SLOT_WIDTH + 2] = xs[0];
    }
  }
}

// One column chunk's share of a 64x64 tile of P = T U_r: with one 64-wide tile
// per block at k <= 64, a tile per workgroup leaves most CUs idle and walks
// all n columns in one chain, so few-block steps split n into chunks of k
// rounded up to 64 columns (the chunks' shares of P then take as much memory
// as T), one workgroup each.  64 columns of T at a time are staged through LDS
// as floats: there the planes of a row-split projection are added in order
// (b0 = 0 tasks also write the sum to T, which then holds U_l^T G whatever the
// cut; no later kernel reads it).  Wave w takes rows 16w .. +15
// of the tile on six bf16 products per fp32 product and writes them to the
// chunk's plane; delta_finish adds the chunks.  tplanes and pplanes: the row
// parts' planes of T and the chunks' planes of P.
// 10 blocks of GPT-2 small (k = 64): 36 -> 20 us with delta_finish; one 2048 x
// 2048 block over 16 row parts: 69 -> 24 us.
constexpr int TSP = 64 + 4;   // LDS pitch of the staged columns of T

__host__ __device__ inline int delta_cols(int k) { return (k + 63) / 64 * 64; }

__device__ __forceinline__ void delta_part(const scao_leaf_desc& L, int a0, int b0, int chunk,
                                           const float* tplanes, float* pplanes,
                                           float (*Ts)[TSP]) {
  const int tid = threadIdx.x, w = tid / 64, l = tid % 64, i = l % 16, g = l / 16;
  const int n = L.n, k = L.k;
  const int parts = SCAO_LF_GET_NSPLIT(L.flags);
  const int64_t tp = plane_floats((int64_t)k * n);
  const int jbeg = chunk * delta_cols(k), jend = min(n, jbeg + delta_cols(k));
  const int dl = b0 + 4 * i;
  int dm = 0;
#pragma unroll
  for (int t = 0; t < 4; ++t) dm |= (dl + t < k) ? (1 << t) : 0;
  v4f acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  for (int jb = jbeg; jb < jend; jb += 64) {
    // rows of U_r past n repeat row n - 1 and meet zeros of T
    v4f cb[2][8];
    if (dm == 15) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          cb[h][e] = gld4(L.Ur + (int64_t)min(jb + 32 * h + 8 * g + e, n - 1) * k + dl);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          cb[h][e] = ldf4(L.Ur, (int64_t)min(jb + 32 * h + 8 * g + e, n - 1) * k + dl, false, dm);
    }
    // 64 columns of T, summed over the row parts: thread -> rows tid / 16 + 16q
    const int col = jb + 4 * (tid % 16);
    int cm = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) cm |= (col + t < n) ? (1 << t) : 0;
    // (rows past k repeat row k - 1: they reach only rows of P past k, which
    // are not stored; no branch between the loads, whose join would wait)
    const float* first = parts > 1 ? tplanes : L.T;
    int64_t at[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) at[q] = (int64_t)min(a0 + tid / 16 + 16 * q, k - 1) * n + col;
    v4f x[4];
    if (cm == 15) {
#pragma unroll
      for (int q = 0; q < 4; ++q) x[q] = gld4(first + at[q]);
#pragma unroll 4
      for (int s = 1; s < parts; ++s)
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] += gld4(first + s * tp + at[q]);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) x[q] = ldf4(first, at[q], false, cm);
      for (int s = 1; s < parts; ++s)
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] += ldf4(first + s * tp, at[q], false, cm);
    }
    if (jb > jbeg) __syncthreads();   // the previous columns' reads
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = tid / 16 + 16 * q, c = a0 + row;
      *(v4f*)&Ts[row][4 * (tid % 16)] = x[q];
      if (parts > 1 && b0 == 0 && c < k && cm)
        stf4(L.T, (int64_t)c * n + col, x[q], cm == 15, cm);
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const v4f lo = *(const v4f*)&Ts[16 * w + i][32 * h + 8 * g];
      const v4f hi = *(const v4f*)&Ts[16 * w + i][32 * h + 8 * g + 4];
      const float xa[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      const bf3 aw = split_bf3(xa);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        float xb[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) xb[e] = cb[h][e][t];
        acc[t] = mfma_x6(aw, split_bf3(xb), acc[t]);
      }
    }
  }
  // element (16w + 4g + r, 4i + t) of the tile
  float* out = pplanes + chunk * plane_floats((int64_t)k * k);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int c = a0 + 16 * w + 4 * g + r;
    if (c < k && dm)
      stf4(out, (int64_t)c * k + dl, v4f{acc[0][r], acc[1][r], acc[2][r], acc[3][r]}, dm == 15,
           dm);
  }
}

// Delta and the natural-norm partial of 16 rows x 64 columns from the chunks'
// shares: one float4 per thread and chunk, eight chunks' loads in flight.
__device__ __forceinline__ void delta_finish(const scao_leaf_desc& L, float eps, int a0, int b0,
                                             const float* pplanes, int slot, double* slots,
                                             double* red) {
  const int tid = threadIdx.x, k = L.k;
  const int chunks = SCAO_LF_GET_DCHUNK(L.flags);
  const int64_t pp = plane_floats((int64_t)k * k);
  const bool sinv4 = L.flags & SCAO_LF_SINV4;
  const int c = a0 + tid / 16, d = b0 + 4 * (tid % 16);
  int dm = 0;
#pragma unroll
  for (int t = 0; t < 4; ++t) dm |= (c < k && d + t < k) ? (1 << t) : 0;
  double nu2 = 0.0;
  if (dm) {
    const float* src = pplanes + (int64_t)c * k + d;
    v4f p = {0.f, 0.f, 0.f, 0.f};
    if (dm == 15) {
      int s = 0;
      for (; s + 8 <= chunks; s += 8) {
        v4f x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = gld4(src + (s + u) * pp);
#pragma unroll
        for (int u = 0; u < 8; ++u) p += x[u];
      }
      for (; s < chunks; ++s) p += gld4(src + s * pp);
    } else {
      for (int s = 0; s < chunks; ++s) p += ldf4(src, s * pp, false, dm);
    }
    const float sl = gld1(L.Sl + c);
    const float sl4 = sinv4 ? sl : inv4(sl);
    const float il2 = sinv4 ? 0.f : inv2(sl, eps);
    v4f o;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float sr = d + t < k ? gld1(L.Sr + d + t) : 1.f;
      o[t] = (sl4 * (sinv4 ? sr : inv4(sr)) - 1.0f) * p[t];
      if (!sinv4 && d + t < k) {
        const float y = (il2 * p[t]) * inv2(sr, eps);
        nu2 += (double)y * (double)y;
      }
    }
    stf4(L.Delta, (int64_t)c * k + d, o, dm == 15, dm);
  }
  if (slot >= 0) {
    double xs[1] = {nu2};
    block_sum<1>(xs, red);
    if (tid == 0) {
      slots[(int64_t)slot * SCAO_SLOT_WIDTH + 0] = 0.0;
      slots[(int64_t)slot * SCAO_SLOT_WIDTH + 1] = 0.0;
      slots[(int64_t)slot * SCAO_SLOT_WIDTH + 2] = xs[0];
    }
  }
}

// A diagonal sub-block of a block-diagonal parameter (SCAO_LF_DIAG: a
// remainder block one row or one column wide, reference
// preconditioner.py:142-153, 232-236).  Nothing is projected: one 64x64 tile
// of it contributes ||g||^2, ||p*decay||^2 (LARS params) and the natural-norm
// sum g^2 / (sqrt(diag) + eps) (:542-544) to the task's slot, in the place
// the projection and delta tasks of a Kronecker block write them.
__device__ __forceinline__ void diag_leaf_reduce(const scao_leaf_desc& L,
                                                 const scao_param_desc& P, int i0, int j0,
                                                 int slot, double* slots, double* red) {
  const int dt = P.dtype;
  const bool decay = P.flags & SCAO_PF_DECAY;
  const bool lars = P.flags & SCAO_PF_LARS;
  double acc[3] = {0.0, 0.0, 0.0};
  // only the elements that are there: the sub-block is one wide, so at most 64
  const int rows = min(64, L.m - i0), cols = min(64, L.n - j0);
  for (int q = threadIdx.x; q < rows * cols; q += 256) {
    const int i = i0 + q / cols, j = j0 + q % cols;
    const int64_t e = L.off + (int64_t)i * L.ld + j;
    const float g = ld1(P.graw, dt, e);
    const float dg = gld1(L.Sl + (int64_t)i * L.n + j);
    acc[0] += (double)(g * g);
    if (lars) {
      const float p = ld1(P.p, dt, e);
      const float pd = decay ? round_to(dt, p * P.decay) : p;
      acc[1] += (double)(pd * pd);
    }
    acc[2] += (double)((g * g) / (sqrtf(dg) + P.eps));
  }
  block_sum<3>(acc, red);
  if (threadIdx.x == 0 && slot >= 0) {
    slots[(int64_t)slot * SCAO_SLOT_WIDTH + 0] = acc[0];
    slots[(int64_t)slot * SCAO_SLOT_WIDTH + 1] = acc[1];
    slots[(int64_t)slot * SCAO_SLOT_WIDTH + 2] = acc[2];
  }
}

// -------------------------------------------------------------- lift ---
// W[i0:i0+64, d0:d0+64] = U_l Delta.  Wave w computes rows i0+16w .. +15.
// On whole columns (k % 16 == 0, d0 + 64 <= k) lane column jj holds
// W columns d0 + 4*jj + t of MFMA tile t, so one float4 of a Delta row feeds
// all four tiles and each row of the result leaves as one float4; the
// reduction runs with NH chunks of operands in flight (fully unrolled for
// k = 16 NC, NC > 0; any multiple of 16 with one chunk of lookahead for
// NC = 0).  Other tiles take the element-wise path.
// W's exact three-way bf16 split (as split_bf3) into the planes h, m, l of
// Wb (plane stride mk elements), at element o: four elements, or one.
__device__ __forceinline__ void split3(float x, __bf16& h, __bf16& m, __bf16& l) {
  h = (__bf16)x;
  const float r = x - (float)h;
  m = (__bf16)r;
  l = (__bf16)(r - (float)m);
}
// four consecutive elements' planes as two packed words each
__device__ __forceinline__ void split4_pk(const v4f& x, v2u& h, v2u& m, v2u& l) {
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    uint32_t a, b, c;
    split3_pk(x[2 * p], x[2 * p + 1], a, b, c);
    h[p] = a;
    m[p] = b;
    l[p] = c;
  }
}
__device__ __forceinline__ void store_split4(uint16_t* wb, int64_t mk, int64_t o, const v4f& x) {
  v2u h, m, l;
  split4_pk(x, h, m, l);
  *(gv2u*)(wb + o) = h;
  *(gv2u*)(wb + mk + o) = m;
  *(gv2u*)(wb + 2 * mk + o) = l;
}
__device__ __forceinline__ void store_split1(uint16_t* wb, int64_t mk, int64_t o, float x) {
  __bf16 h, m, l;
  split3(x, h, m, l);
  ((gu16*)wb)[o] = __builtin_bit_cast(uint16_t, h);
  ((gu16*)wb)[mk + o] = __builtin_bit_cast(uint16_t, m);
  ((gu16*)wb)[2 * mk + o] = __builtin_bit_cast(uint16_t, l);
}

template <int NC>
__device__ __forceinline__ void lift_chunks(const float* __restrict__ urow,
                                            const float* __restrict__ drow, int k,
                                            v4f (&acc)[4]) {
  // urow: U_l row + 4*kk; drow: Delta row 4*kk, columns dl..dl+3
  if constexpr (NC > 0) {
    constexpr int PD = NC < 4 ? NC : 4;
    v4f A[PD], B[PD][4];
#pragma unroll
    for (int d = 0; d < PD; ++d) {
      A[d] = gld4(urow + 16 * d);
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) B[d][s4] = gld4(drow + (int64_t)(16 * d + s4) * (16 * NC));
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d = c % PD;
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma16(A[d][s4], B[d][s4][t], acc[t]);
      if (c + PD < NC) {
        A[d] = gld4(urow + 16 * (c + PD));
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4)
          B[d][s4] = gld4(drow + (int64_t)(16 * (c + PD) + s4) * (16 * NC));
      }
    }
  } else {
    v4f a = gld4(urow), b[4];
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) b[s4] = gld4(drow + (int64_t)s4 * k);
    for (int cb = 0; cb < k; cb += 16) {
      const bool more = cb + 16 < k;
      v4f an = a, bn[4] = {b[0], b[1], b[2], b[3]};
      if (more) {
        an = gld4(urow + cb + 16);
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) bn[s4] = gld4(drow + (int64_t)(cb + 16 + s4) * k);
      }
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma16(a[s4], b[s4][t], acc[t]);
      a = an;
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) b[s4] = bn[s4];
    }
  }
}

__device__ __forceinline__ void lift_tile(const scao_leaf_desc& L, int i0, int d0) {
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  const int m = L.m, k = L.k;
  const int kk = l / 16;
  v4f acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  if (k % 16 == 0 && d0 + 64 <= k) {
    // rows past the block repeat its last one and are not stored
    const int irow = min(i0 + 16 * w + (l % 16), m - 1);
    const int dl = d0 + 4 * (l % 16);
    const float* __restrict__ urow = L.Ul + (int64_t)irow * k + 4 * kk;
    const float* __restrict__ drow = L.Delta + (int64_t)(4 * kk) * k + dl;
    if (k == 256)
      lift_chunks<16>(urow, drow, k, acc);
    else if (k == 128)
      lift_chunks<8>(urow, drow, k, acc);
    else if (k == 64)
      lift_chunks<4>(urow, drow, k, acc);
    else
      lift_chunks<0>(urow, drow, k, acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + 16 * w + 4 * kk + r;
      if (i >= m) continue;
      const int64_t o = (int64_t)i * k + dl;
      const v4f x = v4f{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
      gst4(L.W + o, x);
      if (L.Wb) store_split4(L.Wb, (int64_t)m * k, o, x);
    }
    return;
  }
  const int irow = i0 + 16 * w + (l % 16);
  for (int cb = 0; cb < k; cb += 16) {
    const int c = cb + 4 * kk;
    int cm = 0;
    for (int s = 0; s < 4; ++s) cm |= (c + s < k) ? (1 << s) : 0;
    v4f a = (irow < m && cm) ? ldf4(L.Ul, (int64_t)irow * k + c, cm == 15, cm)
                             : v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int d = d0 + 16 * t + (l % 16);
        const float b = ((cm >> s) & 1) && d < k ? L.Delta[(int64_t)(c + s) * k + d] : 0.f;
        acc[t] = mfma16(a[s], b, acc[t]);
      }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = i0 + 16 * w + 4 * kk + r;
    if (i >= m) continue;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int d = d0 + 16 * t + (l % 16);
      if (d < k) {
        L.W[(int64_t)i * k + d] = acc[t][r];
        if (L.Wb) store_split1(L.Wb, (int64_t)m * k, (int64_t)i * k + d, acc[t][r]);
      }
    }
  }
}

// The same tile for k % 128 == 0 on whole tiles, with the products on
// the bf16 matrix cores (mm64_x6): wave w takes the whole 64 x 64 tile over
// its quarter of k (a multiple of 32), the four partial tiles go through LDS,
// and wave w adds rows 16w .. 16w + 15 of them in order (((w0 + w1) + w2) + w3)
// and writes those rows of W (and Wb).
__device__ __forceinline__ bool lift_x6_ok(const scao_leaf_desc& L, int i0, int d0) {
  return L.k % 128 == 0 && i0 + 64 <= L.m && d0 + 64 <= L.k;
}
__device__ __forceinline__ void lift_tile_x6(const scao_leaf_desc& L, int i0, int d0,
                                             float (*Ps)[64][DP]) {
  const int w = threadIdx.x / 64, l = threadIdx.x % 64, jj = l % 16, g = l / 16;
  const int m = L.m, k = L.k, kq = k / 4;
  v4f acc[4][4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[q][t] = v4f{0.f, 0.f, 0.f, 0.f};
  mm64_x6(L.Ul, k, L.Delta, k, i0, d0, w * kq, w * kq + kq, acc);
  // element (16q + 4g + r, 4jj + t) of the wave's partial tile
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *(v4f*)&Ps[w][16 * q + 4 * g + r][4 * jj] =
          v4f{acc[q][0][r], acc[q][1][r], acc[q][2][r], acc[q][3][r]};
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 16 * w + 4 * g + r;
    const v4f p0 = *(const v4f*)&Ps[0][row][4 * jj];
    const v4f p1 = *(const v4f*)&Ps[1][row][4 * jj];
    const v4f p2 = *(const v4f*)&Ps[2][row][4 * jj];
    const v4f p3 = *(const v4f*)&Ps[3][row][4 * jj];
    v4f x;
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = ((p0[t] + p1[t]) + p2[t]) + p3[t];
    const int64_t o = (int64_t)(i0 + row) * k + d0 + 4 * jj;
    gst4(L.W + o, x);
    if (L.Wb) store_split4(L.Wb, (int64_t)m * k, o, x);
  }
}

// ------------------------------------------------------------- apply ---
// corr[i0:i0+64, j0:j0+64] = W U_r^T; the caller's epilogue consumes it.
// Returns, per lane, corr for rows i0+16w+4*(l/16)+r and columns jl..jl+3.
__device__ __forceinline__ void corr_tile(const scao_leaf_desc& L, int i0, int jl, v4f (&acc)[4]) {
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  const int m = L.m, n = L.n, k = L.k;
  const int kk = l / 16;
  const int irow = i0 + 16 * w + (l % 16);
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  if (k % 16 == 0) {
    // no branch between the loads: rows past the block repeat its last one
    // (they reach only elements past it, which are not stored)
    const float* wrow = L.W + (int64_t)min(irow, m - 1) * k + 4 * kk;
    const float* urow[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) urow[t] = L.Ur + (int64_t)min(jl + t, n - 1) * k + 4 * kk;
    v4f a = gld4(wrow), b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) b[t] = gld4(urow[t]);
    for (int cb = 0; cb < k; cb += 16) {
      const int cn = cb + 16 < k ? cb + 16 : cb;   // the last chunk repeats itself, unused
      const v4f an = gld4(wrow + cn);
      v4f bn[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) bn[t] = gld4(urow[t] + cn);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma16(a[s], b[t][s], acc[t]);
      a = an;
#pragma unroll
      for (int t = 0; t < 4; ++t) b[t] = bn[t];
    }
    return;
  }
  for (int cb = 0; cb < k; cb += 16) {
    const int c = cb + 4 * kk;
    int cm = 0;
    for (int s = 0; s < 4; ++s) cm |= (c + s < k) ? (1 << s) : 0;
    const v4f a = (irow < m && cm) ? ldf4(L.W, (int64_t)irow * k + c, cm == 15, cm)
                                   : v4f{0.f, 0.f, 0.f, 0.f};
    v4f b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int j = jl + t;
      b[t] = (j < n && cm) ? ldf4(L.Ur, (int64_t)j * k + c, cm == 15, cm)
                           : v4f{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t] = mfma16(a[s], b[t][s], acc[t]);
  }
}

}  // namespace

namespace {

// Four consecutive gradient (or parameter) values as loaded by a streaming
// tile: fp32, or (HALF) two words of a 16-bit type, kept raw until the tail
// converts them so that no wait sits between the loads.
template <bool HALF> struct raw4 { typedef v4f type; };
template <> struct raw4<true> { typedef v2u type; };
template <bool HALF>
__device__ __forceinline__ typename raw4<HALF>::type ld_raw4_nt(const void* base, int64_t e) {
  if constexpr (HALF)
    return __builtin_nontemporal_load((const gv2u*)((const uint16_t*)base + e));
  else
    return gld4_nt((const float*)base + e);
}
template <bool HALF>
__device__ __forceinline__ v4f from_raw4(int dt, const typename raw4<HALF>::type& x) {
  if constexpr (HALF)
    return halves_to_v4f(dt, x);
  else
    return x;
}
template <bool HALF>
__device__ __forceinline__ void st_raw4_nt(void* base, int dt, int64_t e, const v4f& x) {
  if constexpr (HALF)
    __builtin_nontemporal_store(v4f_to_halves(dt, x), (gv2u*)((uint16_t*)base + e));
  else
    gst4_nt((float*)base + e, x);
}

// The Phase-2 elementwise tail for one row of four columns (t = 0..3):
// gp = G + corr -> clip -> blend -> Adan moments -> update.  With LARS the
// update itself is returned in `out` (the write waits for the trust ratio);
// otherwise `out` is the new parameter value.  u2 accumulates u^2 over the
// columns in `cmask`.  Operation order and roundings follow
// scao/optimizer.py:584-645 (see the rounding notes on each line).
template <bool GF32, bool LARS>
__device__ __forceinline__ void adan4(const scao_param_desc& P, const scao_param_stat& S, int dt,
                                      const v4f& gr, const v4f& gm, const v4f& corr, v4f& mm,
                                      v4f& vv, v4f& dd, const v4f& pp, const v4f& par, v4f& out,
                                      float& u2, int cmask, bool direct = false) {
  const bool clip = P.flags & SCAO_PF_CLIP;
  const bool gsnr = P.flags & SCAO_PF_GSNR;
  const bool decay = P.flags & SCAO_PF_DECAY;
  const float alpha_nolars = round_to(dt, (float)(-P.lr));
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    // precondition() output in p.dtype; `direct`: corr already is that output
    float gp = round_to(dt, direct ? corr[t] : gr[t] + corr[t]);
    if (clip) gp = round_to(dt, gp * S.clip);           // gp * (tau / nu)
    const float g = GF32 ? gm[t] : gr[t];
    const float geff = P.blend * gp + P.omblend * g;    // b*gp.float() + (1-b)*grad
    const float delta = g - pp[t];
    const float m1 = fmaf(geff, P.omb1, mm[t] * P.beta1);
    const float d1 = fmaf(delta, P.omb3, dd[t] * P.beta3);
    const float gad = geff + P.omb3 * delta;
    const float v1 = fmaf(P.omb2 * gad, gad, vv[t] * P.beta2);
    float x = (m1 / P.bc1 + P.omb3 * (d1 / P.bc3)) / (sqrtf(v1 / P.bc2) + P.eps);
    if (gsnr) x = x * ((fabsf(m1) / (sqrtf(v1) + P.eps)) >= P.gsnr ? 1.0f : 0.0f);
    mm[t] = m1;
    dd[t] = d1;
    vv[t] = v1;
    if (LARS) {
      out[t] = x;
      if (cmask & (1 << t)) u2 = fmaf(x, x, u2);
    } else {
      const float pd = decay ? round_to(dt, par[t] * P.decay) : par[t];
      out[t] = round_to(dt, fmaf(round_to(dt, x), alpha_nolars, pd));
    }
  }
}

__device__ __forceinline__ void write_u2_slot(double* slots, int slot, float u2, double* red) {
  if (slot < 0) return;
  double x[1] = {(double)u2};
  block_sum<1>(x, red);
  if (threadIdx.x == 0) {
    slots[(int64_t)slot * SCAO_SLOT_WIDTH + 0] = 0.0;
    slots[(int64_t)slot * SCAO_SLOT_WIDTH + 1] = 0.0;
    slots[(int64_t)slot * SCAO_SLOT_WIDTH + 2] = x[0];
  }
}

// One 64x64 tile of a block, any shape, dtype or alignment (masked).  Per wave
// 16 rows x 64 columns, 16 elements per lane:
//   1. issue every elementwise load of the tile (g, m, v, d, prev [, p]) --
//      they do not depend on the correction, so HBM latency overlaps step 2;
//   2. corr = W[rows, :] U_r[cols, :]^T on MFMA, with the U_r tile (shared by
//      the four waves) staged once per block through LDS, 64 columns of k at
//      a time;
//   3. the elementwise tail, then the stores.
constexpr int UPAD = 68;   // LDS row pitch (floats) of the staged U_r tile

template <bool GF32, bool LARS>
__device__ __forceinline__ void apply_tile(const scao_leaf_desc& L, const scao_param_desc& P,
                                           const scao_param_stat& S, int i0, int j0, int slot,
                                           double* slots) {
  __shared__ __attribute__((aligned(16))) float Us[64][UPAD];
  __shared__ double red[16];
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  const int m = L.m, n = L.n, k = L.k;
  const int dt = P.dtype;
  const int kk = l / 16;
  const int jl = j0 + 4 * (l % 16);
  int cmask = 15;
  for (int t = 0; t < 4; ++t) cmask = (jl + t < n) ? cmask : (cmask & ~(1 << t));
  const bool vec = cmask == 15;

  // 1) prefetch.  A lane whose four columns all lie in the block loads every
  // row unconditionally, rows past the block from its last one (they are not
  // stored): a branch per load would wait for each.
  v4f gr[4], gm[4], mm[4], vv[4], dd[4], pp[4], par[4];
  int64_t e[4];
  bool rok[4];
  const v4f z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = i0 + 16 * w + 4 * kk + r;
    e[r] = L.off + (int64_t)min(i, m - 1) * L.ld + jl;
    rok[r] = i < m && cmask;
  }
  const bool fused = GF32 && fused_mgrad(P), fmask = GF32 && (P.flags & SCAO_PF_FMASK);
  if (vec) {
    if (dt == SCAO_F32) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        gr[r] = gld4((const float*)P.graw + e[r]);
        if (!LARS) par[r] = gld4((const float*)P.p + e[r]);
      }
    } else {
      v2u hg[4], hp[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        hg[r] = gld2w((const uint16_t*)P.graw + e[r]);
        if (!LARS) hp[r] = gld2w((const uint16_t*)P.p + e[r]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        gr[r] = halves_to_v4f(dt, hg[r]);
        if (!LARS) par[r] = halves_to_v4f(dt, hp[r]);
      }
    }
    // GF32: the fp32 moment buffer, or (fused) the filter's EMA until finish_mgrad
    if (GF32 && (fmask || !fused)) {
      const float* src = fused ? P.fema : (const float*)P.g;
#pragma unroll
      for (int r = 0; r < 4; ++r) gm[r] = gld4(src + e[r]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      mm[r] = gld4(P.exp_avg + e[r]);
      vv[r] = gld4(P.exp_avg_sq + e[r]);
      dd[r] = gld4(P.exp_avg_diff + e[r]);
      pp[r] = gld4(P.prev_grad + e[r]);
    }
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      gr[r] = ld4(P.graw, dt, e[r], false, cmask);
      if (GF32 && (fmask || !fused))
        gm[r] = ldf4(fused ? P.fema : (const float*)P.g, e[r], false, cmask);
      mm[r] = ldf4(P.exp_avg, e[r], false, cmask);
      vv[r] = ldf4(P.exp_avg_sq, e[r], false, cmask);
      dd[r] = ldf4(P.exp_avg_diff, e[r], false, cmask);
      pp[r] = ldf4(P.prev_grad, e[r], false, cmask);
      if (!LARS) par[r] = ld4(P.p, dt, e[r], false, cmask);
    }
  }

  // 2) corr = W U_r^T; for a diagonal sub-block the preconditioned gradient
  //    itself, g / (clamp-free (diag / bias)^(1/4) + 1e-8) (reference
  //    preconditioner.py:506-510), with diag element (i, j) at i*n + j
  v4f acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  const bool dleaf = L.flags & SCAO_LF_DIAG;
  if (dleaf) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (!rok[r]) continue;
      const int i = i0 + 16 * w + 4 * kk + r;
      const v4f dg = ldf4(L.Sl, (int64_t)i * n + jl, false, cmask);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float x = dg[t] / L.dbias;
        const float den = root4(x) + 1e-8f;
        acc[t][r] = gr[r][t] / den;
      }
    }
  }
  // Rows past the block repeat its last ones (their products are not used);
  // columns of k past it (k % 64 != 0) are masked.
  const float* wrow = L.W + (int64_t)min(i0 + 16 * w + (l % 16), m - 1) * k;
  for (int cb0 = 0; cb0 < (dleaf ? 0 : k); cb0 += 64) {
    const int c4 = (threadIdx.x % 16) * 4;
    const bool whole = cb0 + 64 <= k;
    v4f x[4];
    if (whole) {
#pragma unroll
      for (int h = 0; h < 4; ++h)
        x[h] = gld4(L.Ur + (int64_t)min(j0 + (int)threadIdx.x / 16 + 16 * h, n - 1) * k + cb0 + c4);
    } else {
      int mk = 0;
      for (int t = 0; t < 4; ++t) mk |= (cb0 + c4 + t < k) ? (1 << t) : 0;
#pragma unroll
      for (int h = 0; h < 4; ++h)
        x[h] = ldf4(L.Ur, (int64_t)min(j0 + (int)threadIdx.x / 16 + 16 * h, n - 1) * k + cb0 + c4,
                    false, mk);
    }
    v4f a[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = cb0 + 16 * q + 4 * kk;
      if (whole) {
        a[q] = gld4(wrow + c);
      } else {
        int cm = 0;
        for (int s = 0; s < 4; ++s) cm |= (c + s < k) ? (1 << s) : 0;
        a[q] = ldf4(wrow, c, false, cm);
      }
    }
    if (cb0) __syncthreads();
#pragma unroll
    for (int h = 0; h < 4; ++h) *(v4f*)&Us[threadIdx.x / 16 + 16 * h][c4] = x[h];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v4f b[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) b[t] = *(const v4f*)&Us[jl - j0 + t][16 * q + 4 * kk];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma16(a[q][s], b[t][s], acc[t]);
    }
  }

  // 3) elementwise tail
  float u2 = 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (!rok[r]) continue;
    const v4f corr = {acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
    if (GF32 && fused_mgrad(P)) gm[r] = finish_mgrad(P, e[r], gr[r], gm[r], cmask);
    v4f out;
    adan4<GF32, LARS>(P, S, dt, gr[r], gm[r], corr, mm[r], vv[r], dd[r], pp[r], par[r], out, u2,
                      cmask, dleaf);
    stf4(P.exp_avg, e[r], mm[r], vec, cmask);
    stf4(P.exp_avg_sq, e[r], vv[r], vec, cmask);
    stf4(P.exp_avg_diff, e[r], dd[r], vec, cmask);
    stf4(P.prev_grad, e[r], GF32 ? gm[r] : gr[r], vec, cmask);
    st4(LARS ? (void*)P.upd : P.p, dt, e[r], out, vec, cmask);
  }
  write_u2_slot(slots, slot, u2, red);
}

// One 16x256 tile, wholly inside a block of fp32 or (HALF) 16-bit data whose
// rows may start at any element, k % 16 == 0.  (One Llama-1B layer in bf16: 628
// us on masked 64x64 tiles, 423 here; HBM bounds it, 36 B per element.)  A 16-row x 1 KB footprint per block streams
// measurably faster than 64 rows x 256 B.  Wave w owns columns
// j0+64w .. j0+64w+63 of all 16 rows; lane l holds rows i0+4*(l/16)+r and
// columns jl..jl+3, jl = j0+64w+4*(l%16).  The correction for those columns
// needs U_r rows private to the wave, so they are read straight from L2 in
// the MFMA B layout; the 16 rows of W are common to the four waves.
template <bool GF32, bool LARS, bool HALF>
__device__ __forceinline__ void apply_wide(const scao_leaf_desc& L, const scao_param_desc& P,
                                           const scao_param_stat& S, int i0, int j0, int slot,
                                           double* slots) {
  __shared__ double red[16];
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  const int k = L.k;
  const int dt = HALF ? P.dtype : SCAO_F32;
  const int kk = l / 16;
  const int jl = j0 + 64 * w + 4 * (l % 16);

  // 1) the streaming loads (issued in step 2: after the back-projection's
  // operands when k = 64, before them otherwise).  A fused filter's EMA goes
  // first: its keep bits are taken as soon as the back-projection allows,
  // which frees its registers for the rest of the tile.
  typename raw4<HALF>::type gr[4], par[4];
  v4f gm[4], mm[4], vv[4], dd[4], pp[4];
  int64_t e[4];
  const bool fmask = GF32 && (P.flags & SCAO_PF_FMASK);
  auto load_elem = [&]() {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      e[r] = L.off + (int64_t)(i0 + 4 * kk + r) * L.ld + jl;
      if (fmask) gm[r] = gld4_nt(P.fema + e[r]);
      gr[r] = ld_raw4_nt<HALF>(P.graw, e[r]);
      if (GF32 && !fused_mgrad(P)) gm[r] = gld4_nt((const float*)P.g + e[r]);
      mm[r] = gld4_nt(P.exp_avg + e[r]);
      vv[r] = gld4_nt(P.exp_avg_sq + e[r]);
      dd[r] = gld4_nt(P.exp_avg_diff + e[r]);
      pp[r] = gld4_nt(P.prev_grad + e[r]);
      if (!LARS) par[r] = ld_raw4_nt<HALF>(P.p, e[r]);
    }
  };

  // 2) corr = W U_r^T; reduction index c + 4*(l/16) + s for both operands
  v4f acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  const float* __restrict__ wrow = L.W + (int64_t)(i0 + l % 16) * k + 4 * kk;
  const float* __restrict__ urow = L.Ur + (int64_t)jl * k + 4 * kk;
  uint32_t keep = 0xffffu;   // bit 4r+t: the filter keeps element (r, t)
  auto take_keep = [&]() {
    if (fmask) {
      const float thr = *P.fthr;
      keep = 0u;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < 4; ++t) keep |= (gm[r][t] >= thr ? 1u : 0u) << (4 * r + t);
    }
  };
  if (k == 64) {
    // Every operand of the back-projection goes out before the streaming
    // loads and the four chunks run straight-line, so each MFMA waits for its
    // own operands only, not for the streaming loads queued behind them (the
    // vector-memory counter completes in order).  The tile then takes about
    // 170 registers, two waves per SIMD: faster than the streaming loads
    // first at either two or three waves per SIMD (the same sums in the same
    // order).
    v4f A4[4], B4[4][4];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      A4[d] = gld4(wrow + 16 * d);
#pragma unroll
      for (int t = 0; t < 4; ++t) B4[d][t] = gld4(urow + (int64_t)t * 64 + 16 * d);
    }
    load_elem();
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma16(A4[c][s], B4[c][t][s], acc[t]);
    take_keep();
  } else {
    load_elem();
    // operands of chunk c+16 are loaded while chunk c runs on MFMA
    v4f a = gld4(wrow), b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) b[t] = gld4(urow + (int64_t)t * k);
    take_keep();
    for (int c = 0; c < k; c += 16) {
      const bool more = c + 16 < k;
      v4f an = a, bn[4] = {b[0], b[1], b[2], b[3]};
      if (more) {
        an = gld4(wrow + c + 16);
#pragma unroll
        for (int t = 0; t < 4; ++t) bn[t] = gld4(urow + (int64_t)t * k + c + 16);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma16(a[s], b[t][s], acc[t]);
      a = an;
#pragma unroll
      for (int t = 0; t < 4; ++t) b[t] = bn[t];
    }
  }

  // 3) elementwise tail
  float u2 = 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const v4f corr = {acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
    const v4f graw = from_raw4<HALF>(dt, gr[r]);
    const v4f parv = LARS ? v4f{0.f, 0.f, 0.f, 0.f} : from_raw4<HALF>(dt, par[r]);
    if (GF32 && fused_mgrad(P)) gm[r] = finish_mgrad_bits(P, e[r], graw, (keep >> (4 * r)) & 15u, 15);
    v4f out;
    adan4<GF32, LARS>(P, S, dt, graw, gm[r], corr, mm[r], vv[r], dd[r], pp[r], parv, out,
                      u2, 15);
    gst4_nt(P.exp_avg + e[r], mm[r]);
    gst4_nt(P.exp_avg_sq + e[r], vv[r]);
    gst4_nt(P.exp_avg_diff + e[r], dd[r]);
    gst4_nt(P.prev_grad + e[r], GF32 ? gm[r] : graw);
    // the staged update streams past the caches too: it is read back only by
    // k_lars_write, after gigabytes of other traffic, and a caching store
    // evicts the U_r rows the tiles read from L2 (C3 step 12.17 -> 11.98 ms in
    // alternating runs; the strip apply at k = 256 measured slower with it)
    st_raw4_nt<HALF>(LARS ? (void*)P.upd : P.p, dt, e[r], out);
  }
  write_u2_slot(slots, slot, u2, red);
}

// Wide tiles through a two-role pipeline, for ranks where the back-projection
// no longer hides under the streaming of one-tile blocks (k >= 128; at k = 64
// both kernels measure the same).  A block of eight waves takes
// SCAO_APPLY_GROUP consecutive wide tasks.  Waves 0..3 stream tile s (loads,
// Adan tail, stores) between block barriers s and s+1, then issue tile s+1's
// loads.  Waves 4..7 compute corr = W U_r^T into four LDS tile buffers, two
// tiles at a time: tiles 2q and 2q+1 of one column strip share their U_r
// rows, so one pass over them serves both (the operand loads from L2, not
// the MFMAs, bound this role).  Pair q's reduction is split in two halves,
// computed between barriers 2q-2, 2q-1 and 2q, so each barrier interval holds
// one tile's worth of MFMA work; pair 0 is done before barrier 0.  Tiles of
// different blocks or strips, and ranks other than 128 and 256, are computed
// one per half instead.  Each role
// waits only on its own memory operations (the vector-memory counter is in
// order within a wave, so an operand load queued behind the streaming loads
// would wait for them too).  Both roles use apply_wide's lane <-> element
// mapping, so a streaming wave reads exactly the 16x64 slice its partner
// wrote.  u^2 per tile: four wave partials through LDS, summed in a fixed
// order.
constexpr int CP = SCAO_APPLY_WIDE_COLS + 4;   // LDS pitch of a correction row

// One MFMA wave's 16x64 share of corr = W U_r^T: rows of W from wrow, its 64
// U_r rows from urow (lane layout as in apply_wide).  With NC > 0 (k = 16 NC)
// the reduction is fully unrolled with PD chunks of operands in flight, so
// every wait is for one chunk's loads (a loop's back edge makes the compiler
// wait for all of them); NC = 0 takes any multiple of 16 with one chunk of
// lookahead.
template <int NC>
__device__ __forceinline__ void pipe_corr(const float* __restrict__ wrow,
                                          const float* __restrict__ urow, int k, v4f (&acc)[4]) {
  if constexpr (NC > 0) {
    constexpr int PD = 4;
    v4f A[PD], B[PD][4];
#pragma unroll
    for (int d = 0; d < PD && d < NC; ++d) {
      A[d] = gld4(wrow + 16 * d);
#pragma unroll
      for (int t = 0; t < 4; ++t) B[d][t] = gld4(urow + (int64_t)t * (16 * NC) + 16 * d);
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d = c % PD;
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma16(A[d][s4], B[d][t][s4], acc[t]);
      if (c + PD < NC) {
        A[d] = gld4(wrow + 16 * (c + PD));
#pragma unroll
        for (int t = 0; t < 4; ++t) B[d][t] = gld4(urow + (int64_t)t * (16 * NC) + 16 * (c + PD));
      }
    }
  } else {
    v4f a = gld4(wrow), b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) b[t] = gld4(urow + (int64_t)t * k);
    for (int c = 0; c < k; c += 16) {
      const bool more = c + 16 < k;
      v4f an = a, bn[4] = {b[0], b[1], b[2], b[3]};
      if (more) {
        an = gld4(wrow + c + 16);
#pragma unroll
        for (int t = 0; t < 4; ++t) bn[t] = gld4(urow + (int64_t)t * k + c + 16);
      }
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma16(a[s4], b[t][s4], acc[t]);
      a = an;
#pragma unroll
      for (int t = 0; t < 4; ++t) b[t] = bn[t];
    }
  }
}

// The same for two row tiles of one strip (W rows from wa and wb, one U_r
// row set), over NH chunks of a reduction of length K: every U_r load feeds
// both tiles (k = 128 and 256).
// With MID >= 0 a block barrier follows chunk MID's products: the loads of
// the chunks after it are already in flight across the barrier (a block
// barrier waits for LDS operations only), so the second half of a pair starts
// without an operand-latency bubble.
template <int K, int NH, int PD, int MID = -1>
__device__ __forceinline__ void pipe_corr2(const float* __restrict__ wa,
                                           const float* __restrict__ wb,
                                           const float* __restrict__ urow, v4f (&acc)[2][4]) {
  v4f A[PD][2], B[PD][4];
#pragma unroll
  for (int d = 0; d < PD && d < NH; ++d) {
    A[d][0] = gld4(wa + 16 * d);
    A[d][1] = gld4(wb + 16 * d);
#pragma unroll
    for (int t = 0; t < 4; ++t) B[d][t] = gld4(urow + (int64_t)t * K + 16 * d);
  }
#pragma unroll
  for (int c = 0; c < NH; ++c) {
    const int d = c % PD;
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        acc[0][t] = mfma16(A[d][0][s4], B[d][t][s4], acc[0][t]);
        acc[1][t] = mfma16(A[d][1][s4], B[d][t][s4], acc[1][t]);
      }
    if (c + PD < NH) {
      A[d][0] = gld4(wa + 16 * (c + PD));
      A[d][1] = gld4(wb + 16 * (c + PD));
#pragma unroll
      for (int t = 0; t < 4; ++t) B[d][t] = gld4(urow + (int64_t)t * K + 16 * (c + PD));
    }
    if (c == MID) __syncthreads();
  }
}

template <bool GF32, bool LARS>
__global__ __launch_bounds__(512) void k_apply_pipe(const scao_task* __restrict__ tasks, int ntasks,
                                                    const scao_leaf_desc* __restrict__ leaves,
                                                    const scao_param_desc* __restrict__ params,
                                                    const scao_param_stat* __restrict__ stat,
                                                    double* slots) {
  __shared__ __attribute__((aligned(16))) float cbuf[4][16][CP];
  __shared__ double part[2][4];
  const int wv = threadIdx.x / 64, l = threadIdx.x % 64;
  const int w = wv & 3;
  const int kk = l / 16;
  const int t0 = blockIdx.x * SCAO_APPLY_GROUP;
  const int nt = ntasks - t0 < SCAO_APPLY_GROUP ? ntasks - t0 : SCAO_APPLY_GROUP;

  if (wv >= 4) {
    // ---- MFMA role: nt + 1 barriers, as the streaming role ----
    if (nt <= 0) {
      __syncthreads();
      return;
    }
    v4f acc[2][4];
    auto zero = [&]() {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[i][t] = v4f{0.f, 0.f, 0.f, 0.f};
    };
    // tiles 2q and 2q+1 share one pass over their U_r rows
    auto paired = [&](int q) {
      if (2 * q + 1 >= nt) return false;
      const scao_task ta = tasks[t0 + 2 * q], tb = tasks[t0 + 2 * q + 1];
      return tb.idx == ta.idx && tb.b == ta.b && (leaves[ta.idx].k == 256 || leaves[ta.idx].k == 128);
    };
    // a pair's chunks (16 at k = 256, 8 at k = 128), with barrier 2q-1 after
    // the first half when MID
    auto pair = [&](int q, auto mid) {
      const scao_task ta = tasks[t0 + 2 * q], tb = tasks[t0 + 2 * q + 1];
      const scao_leaf_desc& L = leaves[ta.idx];
      const int jl = ta.b + 64 * w + 4 * (l % 16);
      zero();
      if (L.k == 256)
        pipe_corr2<256, 16, 4, decltype(mid)::value>(
            L.W + (int64_t)(ta.a + l % 16) * 256 + 4 * kk,
            L.W + (int64_t)(tb.a + l % 16) * 256 + 4 * kk, L.Ur + (int64_t)jl * 256 + 4 * kk, acc);
      else
        pipe_corr2<128, 8, 4, (decltype(mid)::value < 0 ? -1 : 3)>(
            L.W + (int64_t)(ta.a + l % 16) * 128 + 4 * kk,
            L.W + (int64_t)(tb.a + l % 16) * 128 + 4 * kk, L.Ur + (int64_t)jl * 128 + 4 * kk, acc);
    };
    // otherwise tile 2q in the first half and tile 2q+1 (if any) in the second
    auto single = [&](int q, int h) {
      if (h == 0) zero();
      if (h == 1 && 2 * q + 1 >= nt) return;
      const scao_task tk = tasks[t0 + 2 * q + h];
      const scao_leaf_desc& L = leaves[tk.idx];
      const int k = L.k;
      const int jl = tk.b + 64 * w + 4 * (l % 16);
      const float* __restrict__ wrow = L.W + (int64_t)(tk.a + l % 16) * k + 4 * kk;
      const float* __restrict__ urow = L.Ur + (int64_t)jl * k + 4 * kk;
      if (k == 256)
        pipe_corr<16>(wrow, urow, k, acc[h]);
      else if (k == 128)
        pipe_corr<8>(wrow, urow, k, acc[h]);
      else
        pipe_corr<0>(wrow, urow, k, acc[h]);
    };
    auto put = [&](int q) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int s = 2 * q + i;
        if (s < nt) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            *(v4f*)&cbuf[s & 3][4 * kk + r][64 * w + 4 * (l % 16)] =
                v4f{acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]};
        }
      }
    };
    using NoMid = std::integral_constant<int, -1>;
    using Mid = std::integral_constant<int, 7>;
    if (paired(0)) {
      pair(0, NoMid{});
    } else {
      single(0, 0);
      single(0, 1);
    }
    put(0);
    __syncthreads();                       // barrier 0: tiles 0 and 1 ready
    const int np = (nt + 1) / 2;
    for (int q = 1; q < np; ++q) {
      if (paired(q)) {
        pair(q, Mid{});                    // barrier 2q-1 inside
      } else {
        single(q, 0);
        __syncthreads();                   // barrier 2q-1
        single(q, 1);
      }
      put(q);                              // buffers of tiles 2q-4, 2q-3: consumed
      __syncthreads();                     // barrier 2q: tiles 2q, 2q+1 ready
    }
    for (int b = 2 * np - 1; b < nt + 1; ++b) __syncthreads();
    return;
  }

  // ---- streaming role ----
  v4f gr[4], gm[4], mm[4], vv[4], dd[4], pp[4], par[4];
  int64_t e[4];
  auto prefetch = [&](int s) {
    const scao_task tk = tasks[t0 + s];
    const scao_leaf_desc& L = leaves[tk.idx];
    const scao_param_desc& P = params[L.param];
    const int jl = tk.b + 64 * w + 4 * (l % 16);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      e[r] = L.off + (int64_t)(tk.a + 4 * kk + r) * L.ld + jl;
      gr[r] = gld4_nt((const float*)P.graw + e[r]);
      if (GF32) {
        if (!fused_mgrad(P))
          gm[r] = gld4_nt((const float*)P.g + e[r]);
        else
          gm[r] = (P.flags & SCAO_PF_FMASK) ? gld4_nt(P.fema + e[r]) : gr[r];
      }
      mm[r] = gld4_nt(P.exp_avg + e[r]);
      vv[r] = gld4_nt(P.exp_avg_sq + e[r]);
      dd[r] = gld4_nt(P.exp_avg_diff + e[r]);
      pp[r] = gld4_nt(P.prev_grad + e[r]);
      if (!LARS) par[r] = gld4_nt((const float*)P.p + e[r]);
    }
  };
  auto put_slot = [&](int s) {
    const int slot = tasks[t0 + s].slot;
    if (slot < 0) return;
    const double u2 = ((part[s & 1][0] + part[s & 1][1]) + part[s & 1][2]) + part[s & 1][3];
    slots[(int64_t)slot * SCAO_SLOT_WIDTH + 0] = 0.0;
    slots[(int64_t)slot * SCAO_SLOT_WIDTH + 1] = 0.0;
    slots[(int64_t)slot * SCAO_SLOT_WIDTH + 2] = u2;
  };
  if (nt > 0) prefetch(0);
  for (int s = 0; s < nt; ++s) {
    __syncthreads();     // corr(s) in cbuf[s & 3]; tile s-1's partials in part
    if (s > 0 && w == 0 && l == 0) put_slot(s - 1);
    const scao_task tk = tasks[t0 + s];
    const scao_leaf_desc& L = leaves[tk.idx];
    const scao_param_desc& P = params[L.param];
    const scao_param_stat& S = stat[L.param];
    float u2 = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const v4f corr = *(const v4f*)&cbuf[s & 3][4 * kk + r][64 * w + 4 * (l % 16)];
      if (GF32 && fused_mgrad(P)) gm[r] = finish_mgrad(P, e[r], gr[r], gm[r], 15);
      v4f out;
      adan4<GF32, LARS>(P, S, SCAO_F32, gr[r], gm[r], corr, mm[r], vv[r], dd[r], pp[r], par[r],
                        out, u2, 15);
      gst4_nt(P.exp_avg + e[r], mm[r]);
      gst4_nt(P.exp_avg_sq + e[r], vv[r]);
      gst4_nt(P.exp_avg_diff + e[r], dd[r]);
      gst4_nt(P.prev_grad + e[r], GF32 ? gm[r] : gr[r]);
      if (LARS)
        gst4(P.upd + e[r], out);
      else
        gst4_nt((float*)P.p + e[r], out);
    }
    const double wsum = wave_sum((double)u2);
    if (l == 0) part[s & 1][w] = wsum;
    if (s + 1 < nt) prefetch(s + 1);
  }
  __syncthreads();       // the last tile's partials
  if (nt > 0 && w == 0 && l == 0) put_slot(nt - 1);
}

// ---------------------------------------------- strip-resident apply ---
// Blocks of rank k = 128 or 256.  A task is a run of up to SCAO_APPLY_GROUP
// tiles of one column strip, SW columns x TR rows each (strip_shape: 64 x 128
// at k = 256, 128 x 64 at k = 128), going down the block.  The strip's U_r rows stay in LDS for
// the whole run, so the back-projection reads only W rows from L2 instead of
// every wave refetching U_r per tile.  Per workgroup:
//   waves NS.. (MFMA role): corr(s) = W[rows of tile s, :] U_r[strip, :]^T,
//     32 rows x 64 columns per wave (two 16-row halves sharing each B
//     operand read from LDS), A operands from L2 with chunks of lookahead;
//   waves 0..NS-1 (streaming role, 16 rows x 64 columns each): tile s's loads
//     were issued during tile s-1; once corr(s) is published they run the
//     Phase-2 tail, store, and issue tile s+1's loads.
// The matrix cores and the Phase-2 arithmetic share each SIMD's issue, so the
// products run as six bf16 MFMAs over exact three-way splits (mfma_x6, fp32
// accuracy): W's planes come from scao_kron_lift (Wb), U_r's are split once
// per run into LDS.  Three planes of U_r leave LDS for one correction
// buffer: the streaming waves copy corr(s) to registers and release it (a
// second barrier per tile) before the MFMA waves write corr(s+1).
// Moment gradients (GF): 0, the raw one.  2, the raw one masked by the filter,
// without noise: the filter's averages are loaded ahead of a tile's other
// streams and shrink to one bit per element before the copy of corr takes
// their registers.  1, with noise or from a buffer: no registers are left for
// the copy, so fp32 MFMAs, U_r in LDS as fp32 and two correction buffers (the
// Qwen-3B layer with the filter alone takes 792 us that way, 706 us as 2).
// U_r row r of the strip sits at LDS row 64(r/64) + 16(r%4) + (r%64)/4, so
// that a lane's four B rows (columns 4j + t of its 64-column group) are 16
// rows apart, and the row pitch is 16 bytes past a multiple of 128: a 16-lane
// read phase touches 16 distinct bank groups.
__host__ __device__ constexpr int strip_pitch(int k) { return k + 4 + ((32 - k % 32) % 32); }
__host__ __device__ constexpr int strip_pitch_bf(int k) { return k + 8 + ((64 - k % 64) % 64); }
// Tile shape per rank: SW columns x TR rows (8192 elements), NS = 8
// streaming waves (16 x 64 elements each) and NM = 4 MFMA waves (32 x 64
// each), about 135 KB of LDS: one workgroup per CU.  SW = 64 at k = 256 (what
// LDS holds of U_r), 128 at k = 128: each W row a tile reads then serves 128
// columns.  (64 x 64 tiles at k = 128, two workgroups per CU, measured 10%
// slower: twice the W bytes per element.)
template <int K> struct strip_shape {
  static constexpr int SW = K == 256 ? 64 : 128, TR = 8192 / SW;
  static constexpr int NS = TR * SW / 1024, NM = NS / 2, NT = 64 * (NS + NM);
  // LDS: U_r as three bf16 planes and one correction buffer, or (GF32) as
  // fp32 and two buffers
  static constexpr int lds_bytes(bool bf) {
    return bf ? 3 * SW * strip_pitch_bf(K) * 2 + TR * (SW + 4) * 4
              : SW * strip_pitch(K) * 4 + 2 * TR * (SW + 4) * 4;
  }
};
__device__ __forceinline__ int strip_row(int r) { return 64 * (r / 64) + 16 * (r % 4) + (r % 64) / 4; }

// fp32: corr for rows wa (and wb, 16 rows on) against the LDS strip (lane
// base ub, row pitch pk), k = 16 NC.
template <int NC, int PD>
__device__ __forceinline__ void strip_corr(const float* __restrict__ wa,
                                           const float* __restrict__ wb, const float* ub, int pk,
                                           v4f (&acc)[2][4]) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[h][t] = v4f{0.f, 0.f, 0.f, 0.f};
  v4f A[PD][2], B[2][4];
#pragma unroll
  for (int d = 0; d < PD && d < NC; ++d) {
    A[d][0] = gld4(wa + 16 * d);
    A[d][1] = gld4(wb + 16 * d);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) B[0][t] = *(const v4f*)(ub + 16 * t * pk);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int d = c % PD, cur = c & 1;
    if (c + 1 < NC) {
#pragma unroll
      for (int t = 0; t < 4; ++t) B[cur ^ 1][t] = *(const v4f*)(ub + 16 * t * pk + 16 * (c + 1));
    }
    // chunk c+1's LDS reads go out before chunk c's products (a second
    // register set), so their latency hides behind 32 MFMAs
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        acc[0][t] = mfma16(A[d][0][s4], B[cur][t][s4], acc[0][t]);
        acc[1][t] = mfma16(A[d][1][s4], B[cur][t][s4], acc[1][t]);
      }
    if (c + PD < NC) {
      A[d][0] = gld4(wa + 16 * (c + PD));
      A[d][1] = gld4(wb + 16 * (c + PD));
    }
    // keep chunk c+PD's loads here: the scheduler would otherwise sink
    // them next to their use and expose an L2 round trip per chunk
    __builtin_amdgcn_sched_barrier(0);
  }
}

// bf16 planes: the A operands of one 32-k chunk (both halves, three planes).
struct strip_a {
  bf3 a[2];
};
__device__ __forceinline__ v8bf gld8bf(const uint16_t* p) {
  return __builtin_bit_cast(v8bf, gld4((const float*)p));
}
// wp[h][p]: the lane's row of plane p for half h (column 8*(l/16) included)
__device__ __forceinline__ void strip_load_a(strip_a& A, const uint16_t* const (&wp)[2][3], int c) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    A.a[h].h = gld8bf(wp[h][0] + 32 * c);
    A.a[h].m = gld8bf(wp[h][1] + 32 * c);
    A.a[h].l = gld8bf(wp[h][2] + 32 * c);
  }
}
__device__ __forceinline__ bf3 strip_load_b(const uint16_t* ub, int plane, int pk, int t, int c) {
  const uint16_t* p = ub + 16 * t * pk + 32 * c;
  bf3 b;
  b.h = *(const v8bf*)p;
  b.m = *(const v8bf*)(p + plane);
  b.l = *(const v8bf*)(p + 2 * plane);
  return b;
}

// bf16: corr for the rows of wp (two 16-row halves) against the LDS planes
// (lane base ub, plane stride PLC, row pitch PKC), k = K, with the first PD
// chunks of A already in A[0..PD-1]; the chunk loop is unrolled in
// rotations of PD (every address offset a constant).
template <int K, int PKC, int PLC, int PD>
__device__ __forceinline__ void strip_corr_bf(strip_a (&A)[PD], const uint16_t* const (&wp)[2][3],
                                              const uint16_t* ub, v4f (&acc)[2][4]) {
  constexpr int pk = PKC, plane = PLC, nc = K / 32;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[h][t] = v4f{0.f, 0.f, 0.f, 0.f};
  bf3 B[2];
  B[0] = strip_load_b(ub, plane, pk, 0, 0);
#pragma unroll
  for (int c0 = 0; c0 < nc; c0 += PD) {
#pragma unroll
    for (int d = 0; d < PD; ++d) {
      const int c = c0 + d;
      if (c < nc) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int cur = t & 1;
          if (t < 3)
            B[cur ^ 1] = strip_load_b(ub, plane, pk, t + 1, c);
          else if (c + 1 < nc)
            B[cur ^ 1] = strip_load_b(ub, plane, pk, 0, c + 1);
          // the next B goes out before these products (its own registers)
          __builtin_amdgcn_sched_barrier(0);
          acc[0][t] = mfma_x6(A[d].a[0], B[cur], acc[0][t]);
          acc[1][t] = mfma_x6(A[d].a[1], B[cur], acc[1][t]);
        }
        if (c + PD < nc) strip_load_a(A[d], wp, c + PD);
        // chunk c+PD's loads stay here, PD chunks ahead of their use
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

template <int GF, bool LARS, int K, bool HALF>
__global__ __launch_bounds__(strip_shape<K>::NT) void k_apply_strip(const scao_task* __restrict__ tasks,
                                                     const scao_leaf_desc* __restrict__ leaves,
                                                     const scao_param_desc* __restrict__ params,
                                                     const scao_param_stat* __restrict__ stat,
                                                     double* slots) {
  constexpr bool GF32 = GF != 0, MASK = GF == 2;
  constexpr bool BF = GF != 1;    // bf16 products, one correction buffer
  using SH = strip_shape<K>;
  constexpr int SW = SH::SW, TR = SH::TR, NS = SH::NS, NM = SH::NM;
  constexpr int CB = SW + 4;      // LDS pitch of a correction row
  constexpr int NBUF = BF ? 1 : 2;
  constexpr int CBYTES = NBUF * TR * CB * 4;
  constexpr int LDSB = SH::lds_bytes(BF);
  __shared__ __attribute__((aligned(16))) unsigned char lds[LDSB];
  __shared__ double part[2][NS];
  float(*cbuf)[TR][CB] = (float(*)[TR][CB])(lds + LDSB - CBYTES);
  const int wv = threadIdx.x / 64, l = threadIdx.x % 64;
  const int kk = l / 16;
  const scao_task tk = tasks[blockIdx.x];
  const scao_leaf_desc& L = leaves[tk.idx];
  const int k = L.k;             // == K past the guard below
  constexpr int pk = BF ? strip_pitch_bf(K) : strip_pitch(K);
  const int mw = L.m - L.m % TR;
  int nt = (mw - tk.a) / TR;
  nt = nt < SCAO_APPLY_GROUP ? nt : SCAO_APPLY_GROUP;
  if (nt <= 0) return;   // uniform over the workgroup
  if (k != K || (BF && !L.Wb)) {
    // outside the kernel's contract (the engine never sends this): make the
    // run's norms NaN rather than write anything
    if (threadIdx.x < nt && tk.slot >= 0)
      slots[(int64_t)(tk.slot + threadIdx.x) * SCAO_SLOT_WIDTH + 2] = __builtin_nan("");
    return;
  }

  if (wv >= NS) {
    // ---- MFMA role ----
    constexpr int RP = TR / 32;   // 32-row groups of a tile
    const int mwv = wv - NS, rp = mwv % RP, cg = mwv / RP;
    constexpr int q4 = K / 4;
    auto put = [&](int buf, v4f (&acc)[2][4]) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          *(v4f*)&cbuf[buf][32 * rp + 16 * h + 4 * kk + r][64 * cg + 4 * (l % 16)] =
              v4f{acc[h][0][r], acc[h][1][r], acc[h][2][r], acc[h][3][r]};
    };
    if constexpr (BF) {
      // barriers: A, X_0, then (Y_{s-1}, X_s) for s = 1..nt
      uint16_t* urb = (uint16_t*)lds;
      constexpr int plane = SW * pk;
      for (int q = threadIdx.x - 64 * NS; q < SW * q4; q += 64 * NM) {
        const int r = q / q4, c = q - r * q4;
        const v4f x = gld4(L.Ur + (int64_t)(tk.b + r) * K + 4 * c);
        v2u h, m, lo;
        split4_pk(x, h, m, lo);
        uint16_t* d = urb + strip_row(r) * pk + 4 * c;
        *(v2u*)d = h;
        *(v2u*)(d + plane) = m;
        *(v2u*)(d + 2 * plane) = lo;
      }
      const int64_t mk = (int64_t)L.m * K;
      const uint16_t* ub = urb + (64 * cg + l % 16) * pk + 8 * kk;
      constexpr int PD = K == 256 ? 2 : 3;   // chunks of A lookahead (registers)
      strip_a A[PD];
      const uint16_t* wp[2][3];
      auto rows = [&](int s) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int q = 0; q < 3; ++q)
            wp[h][q] = L.Wb + q * mk + (int64_t)(tk.a + s * TR + 32 * rp + 16 * h + l % 16) * K +
                       8 * kk;
      };
      auto first = [&](int s) {
        rows(s);
#pragma unroll
        for (int d = 0; d < PD; ++d) strip_load_a(A[d], wp, d);
      };
      auto corr = [&](int s, v4f (&acc)[2][4]) {
        strip_corr_bf<K, pk, plane, PD>(A, wp, ub, acc);
      };
      first(0);
      __syncthreads();                                        // A: U_r planes in LDS
      {
        v4f acc[2][4];
        corr(0, acc);
        put(0, acc);
      }
      __syncthreads();                                        // X_0: corr(0) published
      for (int s = 1; s <= nt; ++s) {
        if (s < nt) first(s);                                 // loads in flight across Y
        __syncthreads();                                      // Y_{s-1}: corr(s-1) copied
        if (s < nt) {
          v4f acc[2][4];
          corr(s, acc);
          put(0, acc);
        }
        __syncthreads();                                      // X_s: corr(s) published
      }
    } else {
      // barriers: A, then X_s for s = 0..nt
      float* ur = (float*)lds;
      for (int q = threadIdx.x - 64 * NS; q < SW * q4; q += 64 * NM) {
        const int r = q / q4, c = q - r * q4;
        *(v4f*)&ur[strip_row(r) * pk + 4 * c] = gld4(L.Ur + (int64_t)(tk.b + r) * K + 4 * c);
      }
      __syncthreads();                                        // A: U_r strip in LDS
      const float* ub = &ur[(64 * cg + l % 16) * pk + 4 * kk];
      for (int s = 0; s < nt; ++s) {
        v4f acc[2][4];
        const float* __restrict__ wa =
            L.W + (int64_t)(tk.a + s * TR + 32 * rp + l % 16) * K + 4 * kk;
        const float* __restrict__ wb = wa + (int64_t)16 * K;
        strip_corr<K / 16, 6>(wa, wb, ub, pk, acc);
        put(s & 1, acc);
        __syncthreads();                                      // X_s: corr(s) published
      }
      __syncthreads();                                        // X_nt
    }
    return;
  }

  // ---- streaming role ----
  constexpr int RG = TR / 16;     // 16-row groups of a tile
  const int w = wv, rg = w % RG, cg = w / RG;
  const scao_param_desc& P = params[L.param];
  const scao_param_stat& S = stat[L.param];
  const int dt = HALF ? P.dtype : SCAO_F32;
  typename raw4<HALF>::type gr[4], par[4];
  v4f gm[4], mm[4], vv[4], dd[4], pp[4];
  int64_t e[4];
  const int jc = tk.b + 64 * cg + 4 * (l % 16);
  auto prefetch = [&](int s) {
    if (MASK) {   // first: their bits are taken first
#pragma unroll
      for (int r = 0; r < 4; ++r)
        gm[r] = gld4_nt(P.fema + L.off + (int64_t)(tk.a + s * TR + 16 * rg + 4 * kk + r) * L.ld + jc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      e[r] = L.off + (int64_t)(tk.a + s * TR + 16 * rg + 4 * kk + r) * L.ld + jc;
      gr[r] = ld_raw4_nt<HALF>(P.graw, e[r]);
      if (GF == 1) {
        if (!fused_mgrad(P))
          gm[r] = gld4_nt((const float*)P.g + e[r]);
        else if (P.flags & SCAO_PF_FMASK)
          gm[r] = gld4_nt(P.fema + e[r]);
      }
      mm[r] = gld4_nt(P.exp_avg + e[r]);
      vv[r] = gld4_nt(P.exp_avg_sq + e[r]);
      dd[r] = gld4_nt(P.exp_avg_diff + e[r]);
      pp[r] = gld4_nt(P.prev_grad + e[r]);
      if (!LARS) par[r] = ld_raw4_nt<HALF>(P.p, e[r]);
    }
  };
  auto put_slot = [&](int s) {
    if (tk.slot < 0) return;
    const double* q = part[s & 1];
    double u2 = q[0];
#pragma unroll
    for (int i = 1; i < NS; ++i) u2 += q[i];   // fixed order
    const int64_t slot = tk.slot + s;
    slots[slot * SCAO_SLOT_WIDTH + 0] = 0.0;
    slots[slot * SCAO_SLOT_WIDTH + 1] = 0.0;
    slots[slot * SCAO_SLOT_WIDTH + 2] = u2;
  };
  prefetch(0);
  __syncthreads();                                            // A
  __syncthreads();                                            // X_0: corr(0)
  for (int s = 0; s < nt; ++s) {
    if (s > 0 && w == 0 && l == 0) put_slot(s - 1);
    uint32_t keep = 0u;   // bit 4r+t: the filter keeps element (r, t)
    if (MASK) {
      const float thr = *P.fthr;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < 4; ++t) keep |= (gm[r][t] >= thr ? 1u : 0u) << (4 * r + t);
    }
    v4f cr[4];
    if constexpr (BF) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        cr[r] = *(const v4f*)&cbuf[0][16 * rg + 4 * kk + r][64 * cg + 4 * (l % 16)];
      __syncthreads();                                        // Y_s: the buffer is free
    }
    float u2 = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const v4f corr =
          BF ? cr[r] : *(const v4f*)&cbuf[s & 1][16 * rg + 4 * kk + r][64 * cg + 4 * (l % 16)];
      const v4f graw = from_raw4<HALF>(dt, gr[r]);
      const v4f parv = LARS ? v4f{0.f, 0.f, 0.f, 0.f} : from_raw4<HALF>(dt, par[r]);
      if (MASK) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
          gm[r][t] = graw[t] * (((keep >> (4 * r + t)) & 1u) ? 1.0f : 0.0f);
      } else if (GF32 && fused_mgrad(P)) {
        gm[r] = finish_mgrad(P, e[r], graw, gm[r], 15);
      }
      v4f out;
      adan4<GF32, LARS>(P, S, dt, graw, gm[r], corr, mm[r], vv[r], dd[r], pp[r], parv,
                        out, u2, 15);
      gst4_nt(P.exp_avg + e[r], mm[r]);
      gst4_nt(P.exp_avg_sq + e[r], vv[r]);
      gst4_nt(P.exp_avg_diff + e[r], dd[r]);
      gst4_nt(P.prev_grad + e[r], GF32 ? gm[r] : graw);
      if (LARS && !HALF)
        gst4(P.upd + e[r], out);
      else
        st_raw4_nt<HALF>(LARS ? (void*)P.upd : P.p, dt, e[r], out);
    }
    const double wsum = wave_sum((double)u2);
    if (l == 0) part[s & 1][w] = wsum;
    if (s + 1 < nt) prefetch(s + 1);
    __syncthreads();                                          // X_{s+1}
  }
  if (w == 0 && l == 0) put_slot(nt - 1);
}

// Reference operator: out = G + W U_r^T (dense m x n output), 64 x 64 tiles.
// G's rows go out ahead of the products, whose operands come from L2.
__device__ __forceinline__ void apply_out_tile(const scao_leaf_desc& L, const float* G, float* out, int i0,
                               int j0) {
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  const int m = L.m, n = L.n;
  const int kk = l / 16, jl = j0 + 4 * (l % 16);
  int cmask = 0;
  for (int t = 0; t < 4; ++t) cmask |= (jl + t < n) ? (1 << t) : 0;
  v4f g[4], acc[4];
  // rows past the block repeat its last one and are not stored
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int64_t o = (int64_t)min(i0 + 16 * w + 4 * kk + r, m - 1) * L.ld + jl;
    g[r] = ldf4(G, o, cmask == 15, cmask);
  }
  corr_tile(L, i0, jl, acc);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = i0 + 16 * w + 4 * kk + r;
    if (i >= m || !cmask) continue;
    v4f o;
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] = g[r][t] + acc[t][r];
    stf4(out, (int64_t)i * n + jl, o, cmask == 15, cmask);
  }
}

// The same for 64 rows x 256 columns at k = 64, 64 x 64 per wave: a wave keeps
// its columns' U_r rows in registers for four 16-row tiles, so the operands
// it reads from L2 (32 KB) are half what the tile streams, against two and a
// half times for 16 rows.  Taken from 128 of its tiles, half the CUs, on (whole
// operator, 64 x 64 tiles / this: 64 tiles 31 / 35 us, 128 36 / 38, 225 58 / 53,
// 256 (2048 x 2048) 48 / 42, 1024 101 / 79).  Written for the one width: 64
// registers of U_r rows; at 128 they would be 128 beside the double-buffered W
// and G.
__device__ __forceinline__ void apply_out_wide(const scao_leaf_desc& L, const float* G, float* out,
                                               int i0, int j0) {
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  const int m = L.m, n = L.n;
  const int kk = l / 16, jl = j0 + 64 * w + 4 * (l % 16);
  int cmask = 0;
  for (int t = 0; t < 4; ++t) cmask |= (jl + t < n) ? (1 << t) : 0;
  v4f B[4][4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int t = 0; t < 4; ++t)
      B[d][t] = gld4(L.Ur + (int64_t)min(jl + t, n - 1) * 64 + 4 * kk + 16 * d);
  v4f A[2][4], g[2][4];
  auto load = [&](int q, v4f (&a)[4], v4f (&x)[4]) {
    const float* wrow = L.W + (int64_t)min(i0 + 16 * q + (l % 16), m - 1) * 64 + 4 * kk;
#pragma unroll
    for (int d = 0; d < 4; ++d) a[d] = gld4(wrow + 16 * d);
    if (cmask == 15) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        x[r] = gld4(G + (int64_t)min(i0 + 16 * q + 4 * kk + r, m - 1) * L.ld + jl);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        x[r] = ldf4(G, (int64_t)min(i0 + 16 * q + 4 * kk + r, m - 1) * L.ld + jl, false, cmask);
    }
  };
  load(0, A[0], g[0]);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q < 3) load(q + 1, A[(q + 1) & 1], g[(q + 1) & 1]);   // in flight during the products
    v4f acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma16(A[q & 1][c][s], B[c][t][s], acc[t]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + 16 * q + 4 * kk + r;
      if (i >= m || !cmask) continue;
      v4f o;
#pragma unroll
      for (int t = 0; t < 4; ++t) o[t] = g[q & 1][r][t] + acc[t][r];
      stf4(out, (int64_t)i * n + jl, o, cmask == 15, cmask);
    }
  }
}

// ---------------------------------------------------------- kernels ---
template <bool DO_P, int CR, int NT, int DT, bool EDGE>
__global__ __launch_bounds__(NT) void k_project(const scao_task* __restrict__ tasks,
                                                const scao_leaf_desc* __restrict__ leaves,
                                                const scao_param_desc* __restrict__ params,
                                                double* slots) {
  const scao_task tk = tasks[blockIdx.x];
  const scao_leaf_desc L = leaves[tk.idx];
  __shared__ __attribute__((aligned(16))) project_lds<CR> lds;
  project_part<DO_P, CR, NT, DT, EDGE>(lds, L, params[L.param], tk.a, tk.b, tk.slot, slots);
}
// two waves per SIMD: the bf16-product tiles fit 256 registers without spilling
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_delta(
    const scao_task* __restrict__ tasks, const scao_leaf_desc* __restrict__ leaves,
    const scao_param_desc* __restrict__ params, double* slots) {
  const scao_task tk = tasks[blockIdx.x];
  const scao_leaf_desc L = leaves[tk.idx];
  __shared__ __attribute__((aligned(16))) float Ps[3][64][DP];
  __shared__ double red[16];
  if (L.flags & SCAO_LF_DIAG) {
    diag_leaf_reduce(L, params[L.param], tk.a, tk.b, tk.slot, slots, red);
    return;
  }
  if (SCAO_LF_GET_DCHUNK(L.flags)) {
    delta_finish(L, params[L.param].eps, tk.a, tk.b,
                 L.Delta + plane_floats((int64_t)L.k * L.k), tk.slot, slots, red);
    return;
  }
  const bool fast = tk.a + 64 <= L.k && tk.b + 64 <= L.k && (L.n % 64 == 0);
  if (fast && L.n % 128 == 0)
    delta_tile<true, true>(L, params[L.param].eps, tk.a, tk.b, tk.slot, slots, Ps, red);
  else if (fast)
    delta_tile<true>(L, params[L.param].eps, tk.a, tk.b, tk.slot, slots, Ps, red);
  else
    delta_tile<false>(L, params[L.param].eps, tk.a, tk.b, tk.slot, slots, Ps, red);
}
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_delta_part(
    const scao_task* __restrict__ tasks, const scao_leaf_desc* __restrict__ leaves) {
  __shared__ __attribute__((aligned(16))) float Ts[64][TSP];
  const scao_task tk = tasks[blockIdx.x];
  const scao_leaf_desc L = leaves[tk.idx];
  // a leaf without column chunks has no planes to write
  if ((unsigned)(tk.b >> 16) >= (unsigned)SCAO_LF_GET_DCHUNK(L.flags)) return;
  delta_part(L, tk.a, tk.b & 0xffff, tk.b >> 16, L.T + plane_floats((int64_t)L.k * L.n),
             L.Delta + plane_floats((int64_t)L.k * L.k), Ts);
}
// two waves per SIMD: the bf16-product tiles fit 256 registers without spilling
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_lift(
    const scao_task* __restrict__ tasks, const scao_leaf_desc* __restrict__ leaves) {
  __shared__ __attribute__((aligned(16))) float Ps[4][64][DP];
  const scao_task tk = tasks[blockIdx.x];
  const scao_leaf_desc L = leaves[tk.idx];
  if (lift_x6_ok(L, tk.a, tk.b))
    lift_tile_x6(L, tk.a, tk.b, Ps);
  else
    lift_tile(L, tk.a, tk.b);
}
template <bool GF32, bool LARS, bool FAST, bool HALF = false>
__global__ __launch_bounds__(256) void k_apply(const scao_task* __restrict__ tasks,
                                               const scao_leaf_desc* __restrict__ leaves,
                                               const scao_param_desc* __restrict__ params,
                                               const scao_param_stat* __restrict__ stat,
                                               double* slots) {
  const scao_task tk = tasks[blockIdx.x];
  const scao_leaf_desc L = leaves[tk.idx];
  if (FAST)
    apply_wide<GF32, LARS, HALF>(L, params[L.param], stat[L.param], tk.a, tk.b, tk.slot, slots);
  else
    apply_tile<GF32, LARS>(L, params[L.param], stat[L.param], tk.a, tk.b, tk.slot, slots);
}

// single-block reference operator (descriptors by value, tiles from blockIdx)
template <int CR, int NT>
__global__ __launch_bounds__(NT) void k_project_one(scao_leaf_desc L, scao_param_desc P,
                                                    float* tplanes) {
  __shared__ __attribute__((aligned(16))) project_lds<CR> lds;
  const int strips = (L.n + SCAO_PROJ_COLS - 1) / SCAO_PROJ_COLS, kt = (L.k + CR - 1) / CR;
  const int j0 = (int)(blockIdx.x % strips) * SCAO_PROJ_COLS;
  const int c0 = (int)(blockIdx.x / strips % kt) * CR, part = (int)(blockIdx.x / (strips * kt));
  const int parts = SCAO_LF_GET_NSPLIT(L.flags), rows = split_rows(L.m, parts);
  const int i_beg = part * rows, i_end = min(L.m, i_beg + rows);
  float* T = parts > 1 ? tplanes + part * plane_floats((int64_t)L.k * L.n) : L.T;
  const bool whole = j0 + SCAO_PROJ_COLS <= L.n && (i_end - i_beg) % PR == 0 &&
                     L.ld < SHORT_ROWS;
  if (whole && c0 + CR <= L.k)
    project_tile<false, CR, NT, SCAO_F32, false>(lds, L, P, j0, c0, i_beg, i_end, T, -1, nullptr);
  else if (whole)
    project_tile<false, CR, NT, SCAO_F32, false, true>(lds, L, P, j0, c0, i_beg, i_end, T, -1, nullptr);
  else
    project_tile<false, CR, NT, SCAO_F32, true>(lds, L, P, j0, c0, i_beg, i_end, T, -1, nullptr);
}
__global__ __launch_bounds__(256) void k_delta_one(scao_leaf_desc L) {
  __shared__ __attribute__((aligned(16))) float Ps[3][64][DP];
  __shared__ double red[16];
  const int tiles = (L.k + 63) / 64;
  delta_tile<false>(L, 1e-8f, (blockIdx.x / tiles) * 64, (blockIdx.x % tiles) * 64, -1, nullptr,
                    Ps, red);
}
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_delta_part_one(scao_leaf_desc L, const float* tplanes,
                                                        float* pplanes) {
  __shared__ __attribute__((aligned(16))) float Ts[64][TSP];
  const int tiles = (L.k + 63) / 64, tile = (int)blockIdx.x % (tiles * tiles);
  delta_part(L, (tile / tiles) * 64, (tile % tiles) * 64, (int)blockIdx.x / (tiles * tiles),
             tplanes, pplanes, Ts);
}
__global__ __launch_bounds__(256) void k_delta_finish_one(scao_leaf_desc L, const float* pplanes) {
  __shared__ double red[16];
  const int tiles = (L.k + 63) / 64;
  delta_finish(L, 1e-8f, ((int)blockIdx.x / tiles) * 16, ((int)blockIdx.x % tiles) * 64, pplanes,
               -1, nullptr, red);
}
__global__ __launch_bounds__(256) void k_lift_one(scao_leaf_desc L) {
  const int tiles = (L.k + 63) / 64;
  lift_tile(L, (blockIdx.x / tiles) * 64, (blockIdx.x % tiles) * 64);
}
__global__ __launch_bounds__(256) void k_apply_out_one(scao_leaf_desc L, const float* G,
                                                      float* out) {
  const int tiles = (L.n + 63) / 64;
  apply_out_tile(L, G, out, (blockIdx.x / tiles) * 64, (blockIdx.x % tiles) * 64);
}
__global__ __launch_bounds__(256) void k_apply_out_wide(scao_leaf_desc L, const float* G,
                                                       float* out) {
  const int tiles = (L.n + 255) / 256;
  apply_out_wide(L, G, out, (blockIdx.x / tiles) * 64, (blockIdx.x % tiles) * 256);
}

template <int GF, bool LARS, int K, class... A>
void launch_strip_gf(bool half, dim3 g, hipStream_t s, A... args) {
  if (half)
    hipLaunchKernelGGL((k_apply_strip<GF, LARS, K, true>), g, dim3(strip_shape<K>::NT), 0, s,
                       args...);
  else
    hipLaunchKernelGGL((k_apply_strip<GF, LARS, K, false>), g, dim3(strip_shape<K>::NT), 0, s,
                       args...);
}
template <bool LARS, int K, class... A>
void launch_strip(int gf, bool half, dim3 g, hipStream_t s, A... args) {
  if (gf == 0)
    launch_strip_gf<0, LARS, K>(half, g, s, args...);
  else if (gf == 1)
    launch_strip_gf<1, LARS, K>(half, g, s, args...);
  else
    launch_strip_gf<2, LARS, K>(half, g, s, args...);
}
// whole projection tiles of the data type: 0 fp32, 1 bf16, 2 fp16
template <bool DO_P, int CR, int NT>
void launch_project(int type, dim3 g, hipStream_t s, const scao_task* tasks,
                    const scao_leaf_desc* leaves, const scao_param_desc* params, double* slots) {
  if (type == 0)
    hipLaunchKernelGGL((k_project<DO_P, CR, NT, SCAO_F32, false>), g, dim3(NT), 0, s, tasks,
                       leaves, params, slots);
  else if (type == 1)
    hipLaunchKernelGGL((k_project<DO_P, CR, NT, SCAO_BF16, false>), g, dim3(NT), 0, s, tasks,
                       leaves, params, slots);
  else
    hipLaunchKernelGGL((k_project<DO_P, CR, NT, SCAO_F16, false>), g, dim3(NT), 0, s, tasks,
                       leaves, params, slots);
}

}  // namespace

// ------------------------------------------------------------- C ABI ---
extern "C" int scao_kron_project(const scao_task* tasks, int ntasks, const scao_leaf_desc* leaves,
                                 const scao_param_desc* params, double* slots, int variant,
                                 void* stream) {
  SCAO_CHECK_ARG(ntasks >= 0, "scao_kron_project: ntasks < 0");
  if (ntasks == 0) return SCAO_OK;
  SCAO_CHECK_ARG(tasks && leaves && params && slots, "scao_kron_project: null pointer");
  const int width = (variant >> 2) & 3, type = (variant >> 4) & 3;
  SCAO_CHECK_ARG(variant >= 0 && variant < 64 && width < 3 && type < 3 &&
                     ((variant & 1) || variant < 4),
                 "scao_kron_project: bad variant %d", variant);
  hipStream_t s = (hipStream_t)stream;
  const dim3 g(ntasks);
  if (!(variant & 1)) {
    if (variant & 2)
      hipLaunchKernelGGL((k_project<true, 64, 256, SCAO_F32, true>), g, dim3(256), 0, s, tasks,
                         leaves, params, slots);
    else
      hipLaunchKernelGGL((k_project<false, 64, 256, SCAO_F32, true>), g, dim3(256), 0, s, tasks,
                         leaves, params, slots);
  } else if (variant & 2) {
    switch (width) {
      case 0: launch_project<true, 64, 256>(type, g, s, tasks, leaves, params, slots); break;
      case 1: launch_project<true, 128, 512>(type, g, s, tasks, leaves, params, slots); break;
      default: launch_project<true, 256, 512>(type, g, s, tasks, leaves, params, slots); break;
    }
  } else {
    switch (width) {
      case 0: launch_project<false, 64, 256>(type, g, s, tasks, leaves, params, slots); break;
      case 1: launch_project<false, 128, 512>(type, g, s, tasks, leaves, params, slots); break;
      default: launch_project<false, 256, 512>(type, g, s, tasks, leaves, params, slots); break;
    }
  }
  SCAO_LAUNCH_CHECK("scao_kron_project");
  return SCAO_OK;
}

extern "C" int scao_kron_delta(const scao_task* tasks, int ntasks, const scao_leaf_desc* leaves,
                               const scao_param_desc* params, double* slots, void* stream) {
  SCAO_CHECK_ARG(ntasks >= 0, "scao_kron_delta: ntasks < 0");
  if (ntasks == 0) return SCAO_OK;
  SCAO_CHECK_ARG(tasks && leaves && params && slots, "scao_kron_delta: null pointer");
  hipLaunchKernelGGL(k_delta, dim3(ntasks), dim3(256), 0, (hipStream_t)stream, tasks, leaves,
                     params, slots);
  SCAO_LAUNCH_CHECK("scao_kron_delta");
  return SCAO_OK;
}

extern "C" int scao_kron_delta_part(const scao_task* tasks, int ntasks,
                                    const scao_leaf_desc* leaves, void* stream) {
  SCAO_CHECK_ARG(ntasks >= 0, "scao_kron_delta_part: ntasks < 0");
  if (ntasks == 0) return SCAO_OK;
  SCAO_CHECK_ARG(tasks && leaves, "scao_kron_delta_part: null pointer");
  hipLaunchKernelGGL(k_delta_part, dim3(ntasks), dim3(256), 0, (hipStream_t)stream, tasks, leaves);
  SCAO_LAUNCH_CHECK("scao_kron_delta_part");
  return SCAO_OK;
}

extern "C" int scao_kron_lift(const scao_task* tasks, int ntasks, const scao_leaf_desc* leaves,
                              void* stream) {
  SCAO_CHECK_ARG(ntasks >= 0, "scao_kron_lift: ntasks < 0");
  if (ntasks == 0) return SCAO_OK;
  SCAO_CHECK_ARG(tasks && leaves, "scao_kron_lift: null pointer");
  hipLaunchKernelGGL(k_lift, dim3(ntasks), dim3(256), 0, (hipStream_t)stream, tasks, leaves);
  SCAO_LAUNCH_CHECK("scao_kron_lift");
  return SCAO_OK;
}

extern "C" int scao_kron_apply(const scao_task* tasks, int ntasks, const scao_leaf_desc* leaves,
                               const scao_param_desc* params, const scao_param_stat* stat,
                               double* slots, int variant, void* stream) {
  SCAO_CHECK_ARG(ntasks >= 0, "scao_kron_apply: ntasks < 0");
  if (ntasks == 0) return SCAO_OK;
  SCAO_CHECK_ARG(tasks && leaves && params && stat && slots, "scao_kron_apply: null pointer");
  const bool half = variant & 64, mask = variant & 128;
  SCAO_CHECK_ARG(variant >= 0 && variant < 256 && ((variant & ~3) == 0 || (variant & 4)) &&
                     !(half && (variant & 8)) && (!mask || (variant & 17) == 17) &&
                     (!(variant & 32) || (variant & 24)),
                 "scao_kron_apply: bad variant %d", variant);
  hipStream_t s = (hipStream_t)stream;
  if (variant & 16) {
    const dim3 gs(ntasks);
    const int gf = mask ? 2 : variant & 1;
    if (variant & 32) {
      if (variant & 2)
        launch_strip<true, 128>(gf, half, gs, s, tasks, leaves, params, stat, slots);
      else
        launch_strip<false, 128>(gf, half, gs, s, tasks, leaves, params, stat, slots);
    } else {
      if (variant & 2)
        launch_strip<true, 256>(gf, half, gs, s, tasks, leaves, params, stat, slots);
      else
        launch_strip<false, 256>(gf, half, gs, s, tasks, leaves, params, stat, slots);
    }
    SCAO_LAUNCH_CHECK("scao_kron_apply");
    return SCAO_OK;
  }
  if (variant & 8) {
    const dim3 gp((ntasks + SCAO_APPLY_GROUP - 1) / SCAO_APPLY_GROUP), bp(512);
#define SCAO_APPLY_PIPE(GF, LA) \
  hipLaunchKernelGGL((k_apply_pipe<GF, LA>), gp, bp, 0, s, tasks, ntasks, leaves, params, stat, slots)
    switch (variant & 3) {
      case 0: SCAO_APPLY_PIPE(false, false); break;
      case 1: SCAO_APPLY_PIPE(true, false); break;
      case 2: SCAO_APPLY_PIPE(false, true); break;
      default: SCAO_APPLY_PIPE(true, true); break;
    }
#undef SCAO_APPLY_PIPE
    SCAO_LAUNCH_CHECK("scao_kron_apply");
    return SCAO_OK;
  }
  dim3 g(ntasks), b(256);
#define SCAO_APPLY(...) \
  hipLaunchKernelGGL((k_apply<__VA_ARGS__>), g, b, 0, s, tasks, leaves, params, stat, slots)
  switch (variant) {
    case 0: SCAO_APPLY(false, false, false); break;
    case 1: SCAO_APPLY(true, false, false); break;
    case 2: SCAO_APPLY(false, true, false); break;
    case 3: SCAO_APPLY(true, true, false); break;
    case 4: SCAO_APPLY(false, false, true); break;
    case 5: SCAO_APPLY(true, false, true); break;
    case 6: SCAO_APPLY(false, true, true); break;
    case 7: SCAO_APPLY(true, true, true); break;
    case 68: SCAO_APPLY(false, false, true, true); break;
    case 69: SCAO_APPLY(true, false, true, true); break;
    case 70: SCAO_APPLY(false, true, true, true); break;
    case 71: SCAO_APPLY(true, true, true, true); break;
    default: SCAO_CHECK_ARG(false, "scao_kron_apply: bad variant %d", variant);
  }
#undef SCAO_APPLY
  SCAO_LAUNCH_CHECK("scao_kron_apply");
  return SCAO_OK;
}

extern "C" int64_t scao_fused_kronecker_workspace(int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  return (k * n + k * k + m * k) * (int64_t)sizeof(float);
}

namespace {

// The launches of the reference operator over one block (project, delta in one
// or two, lift, apply), with the block's T, Delta and W in the k*n + k*k + m*k
// floats at ws.
int launch_fused_kronecker(const float* U_l, const float* s_l_inv4, const float* U_r,
                           const float* s_r_inv4, const float* G, int64_t ldG, float* out,
                           int64_t m, int64_t n, int64_t k, float* ws, hipStream_t s) {
  scao_leaf_desc L = {};
  L.Ul = U_l;
  L.Ur = U_r;
  L.Sl = s_l_inv4;
  L.Sr = s_r_inv4;
  L.T = ws;
  L.Delta = ws + k * n;
  L.W = ws + k * n + k * k;
  L.off = 0;
  L.ld = ldG;
  L.param = 0;
  L.m = (int)m;
  L.n = (int)n;
  L.k = (int)k;
  L.flags = SCAO_LF_SINV4;
  scao_param_desc P = {};
  P.g = G;
  P.graw = G;
  P.dtype = SCAO_F32;
  // One block's strips are far fewer than the CUs, so the rows are split too
  // (at least 128 per part, up to a workgroup per CU) and P is formed by column
  // chunks.  Their planes of T and P live in `out`, which the last launch
  // overwrites, so the scratch stays T, Delta and W.  An `out` that shares
  // storage with G, U_l, s_l or s_r, which are still read while the planes are
  // written, or has no room for the planes takes fewer parts or none.
  // 2048 x 2048 at k = 64: projection 337 -> 13 us, P 69 -> 24 us.
  const int64_t strips = (n + SCAO_PROJ_COLS - 1) / SCAO_PROJ_COLS;
  const int cr = k > 128 ? 256 : k > 64 ? 128 : 64;
  const int64_t kt = (k + cr - 1) / cr, pt = (k + 63) / 64;
  const int64_t tp = plane_floats(k * n), pp = plane_floats(k * k);
  int64_t chunks = (n + delta_cols((int)k) - 1) / delta_cols((int)k);
  auto clear_of_out = [&](const float* p, int64_t floats) {
    return (uintptr_t)out >= (uintptr_t)(p + floats) || (uintptr_t)(out + m * n) <= (uintptr_t)p;
  };
  const bool apart = clear_of_out(G, (m - 1) * ldG + n) && clear_of_out(U_l, m * k) &&
                     clear_of_out(s_l_inv4, k) && clear_of_out(s_r_inv4, k);
  const int64_t room = apart ? m * n : 0;
  if (chunks > 255 || chunks * pp > room) chunks = 0;
  int64_t parts = 1;
  if (chunks) {
    parts = std::min<int64_t>(std::min<int64_t>(m / 128, 256 / (strips * kt)),
                              std::min<int64_t>(64, (room - chunks * pp) / tp));
    parts = parts > 1 ? (m + split_rows((int)m, (int)parts) - 1) / split_rows((int)m, (int)parts) : 1;
  }
  L.flags |= (int)(parts << SCAO_LF_NSPLIT_SHIFT) | (int)(chunks << SCAO_LF_DCHUNK_SHIFT);
  float* tplanes = out;
  float* pplanes = out + (parts > 1 ? parts * tp : 0);
  const dim3 gp((unsigned)(strips * kt * parts));
  if (cr == 256)
    hipLaunchKernelGGL((k_project_one<256, 512>), gp, dim3(512), 0, s, L, P, tplanes);
  else if (cr == 128)
    hipLaunchKernelGGL((k_project_one<128, 512>), gp, dim3(512), 0, s, L, P, tplanes);
  else
    hipLaunchKernelGGL((k_project_one<64, 256>), gp, dim3(256), 0, s, L, P, tplanes);
  SCAO_LAUNCH_CHECK("scao_fused_kronecker_precond/project");
  if (chunks) {
    hipLaunchKernelGGL(k_delta_part_one, dim3((unsigned)(pt * pt * chunks)), dim3(256), 0, s, L,
                       tplanes, pplanes);
    SCAO_LAUNCH_CHECK("scao_fused_kronecker_precond/delta part");
    hipLaunchKernelGGL(k_delta_finish_one, dim3((unsigned)((k + 15) / 16 * pt)), dim3(256), 0, s, L,
                       pplanes);
  } else {
    hipLaunchKernelGGL(k_delta_one, dim3((unsigned)(pt * pt)), dim3(256), 0, s, L);
  }
  SCAO_LAUNCH_CHECK("scao_fused_kronecker_precond/delta");
  const int kt64 = (int)pt;
  hipLaunchKernelGGL(k_lift_one, dim3((int)((m + 63) / 64) * kt64), dim3(256), 0, s, L);
  SCAO_LAUNCH_CHECK("scao_fused_kronecker_precond/lift");
  const int64_t wide = (m + 63) / 64 * ((n + 255) / 256);
  if (k == 64 && wide >= 128)
    hipLaunchKernelGGL(k_apply_out_wide, dim3((unsigned)wide), dim3(256), 0, s, L, G, out);
  else
    hipLaunchKernelGGL(k_apply_out_one, dim3((int)((m + 63) / 64) * (int)((n + 63) / 64)),
                       dim3(256), 0, s, L, G, out);
  SCAO_LAUNCH_CHECK("scao_fused_kronecker_precond/apply");
  return SCAO_OK;
}

// Scratch of the no-allocation entry point: one copy per GPU, alive until the
// process ends.  Host code never uses the array's name as an address (on the
// host it is only a stand-in for the symbol): each device's address comes
// from hipGetSymbolAddress, fetched once with that device current.
static __device__ __align__(256) float scratch[SCAO_NOALLOC_SCRATCH_BYTES / sizeof(float)];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kMaxDevices] = {};

// The array of the current device, which must be the device of `stream` (a
// non-null stream of another GPU is rejected: its kernels would be handed an
// address in the wrong GPU's copy).
int scratch_for_current_device(hipStream_t stream, float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    scao_set_error("scao_fused_kronecker_precond_noalloc: hipGetDevice: %s", hipGetErrorString(e));
    return SCAO_ERR_HIP;
  }
  if (stream) {
    hipDevice_t sdev = -1;
    e = hipStreamGetDevice(stream, &sdev);
    if (e != hipSuccess) {
      scao_set_error("scao_fused_kronecker_precond_noalloc: hipStreamGetDevice: %s",
                     hipGetErrorString(e));
      return SCAO_ERR_HIP;
    }
    if ((int)sdev != dev) {
      scao_set_error("scao_fused_kronecker_precond_noalloc: stream of device %d while device %d "
                     "is current (make the stream's device current)", (int)sdev, dev);
      return SCAO_ERR_INVALID;
    }
  }
  if (dev < 0 || dev >= kMaxDevices) {
    scao_set_error("scao_fused_kronecker_precond_noalloc: device %d out of range", dev);
    return SCAO_ERR_INVALID;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      scao_set_error("scao_fused_kronecker_precond_noalloc: hipGetSymbolAddress: %s",
                     hipGetErrorString(e));
      return SCAO_ERR_HIP;
    }
    g_scratch_ptr[dev] = (float*)p;
  }
  *out = g_scratch_ptr[dev];
  return SCAO_OK;
}

}  // namespace

#define SCAO_FUSED_ARGS_CHECK(name)                                                          \
  SCAO_CHECK_ARG(U_l && s_l_inv4 && U_r && s_r_inv4 && G && out, name ": null pointer");   \
  SCAO_CHECK_ARG(m > 0 && n > 0 && k > 0 && ldG >= n,                                      \
                 name ": bad shape m=%lld n=%lld k=%lld ldG=%lld", (long long)m,           \
                 (long long)n, (long long)k, (long long)ldG);                              \
  SCAO_CHECK_ARG(m < (1LL << 31) && n < (1LL << 31) && k <= 4096, name ": dimension too large")

extern "C" int scao_fused_kronecker_precond(const float* U_l, const float* s_l_inv4,
                                            const float* U_r, const float* s_r_inv4,
                                            const float* G, int64_t ldG, float* out, int64_t m,
                                            int64_t n, int64_t k, void* workspace,
                                            void* stream) {
  SCAO_CHECK_ARG(workspace, "scao_fused_kronecker_precond: null pointer");
  SCAO_FUSED_ARGS_CHECK("scao_fused_kronecker_precond");
  return launch_fused_kronecker(U_l, s_l_inv4, U_r, s_r_inv4, G, ldG, out, m, n, k,
                                (float*)workspace, (hipStream_t)stream);
}

extern "C" int scao_fused_kronecker_precond_noalloc(const float* U_l, const float* s_l_inv4,
                                                    const float* U_r, const float* s_r_inv4,
                                                    const float* G, int64_t ldG, float* out,
                                                    int64_t m, int64_t n, int64_t k,
                                                    void* stream) {
  SCAO_FUSED_ARGS_CHECK("scao_fused_kronecker_precond_noalloc");
  const int64_t need = scao_fused_kronecker_workspace(m, n, k);
  SCAO_CHECK_ARG(need <= (int64_t)SCAO_NOALLOC_SCRATCH_BYTES,
                 "scao_fused_kronecker_precond_noalloc: m=%lld n=%lld k=%lld needs %lld bytes "
                 "of scratch, above the %lld-byte maximum (use scao_fused_kronecker_precond "
                 "with a workspace)",
                 (long long)m, (long long)n, (long long)k, (long long)need,
                 (long long)SCAO_NOALLOC_SCRATCH_BYTES);
  float* ws = nullptr;
  const int rc = scratch_for_current_device((hipStream_t)stream, &ws);
  if (rc != SCAO_OK) return rc;
  return launch_fused_kronecker(U_l, s_l_inv4, U_r, s_r_inv4, G, ldG, out, m, n, k, ws,
                                (hipStream_t)stream);
}
