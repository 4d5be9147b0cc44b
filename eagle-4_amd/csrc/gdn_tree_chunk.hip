// GDN tree chunk form on the gfx950 matrix cores (kernels/gdn_tree_records.py:276-361, 496-579): the records
// contract's verify without per-node rounding, solved in closed form per (request, value head) instead of walked node
// by node (trees of at most 16 nodes first; gdn_chunk_wide_kernel takes up to 64):
//
//   R = strict-ancestor closure of the parent links,   G_t = product of exp(g) along t's root path,
//   L = diag(beta) (R o G_t/G_j o K K^T),               D = (I + L)^-1 diag(beta) (V - diag(G) K S0^T),
//   O = diag(G) Q S0^T + ((R + I) o G_t/G_j o Q K^T) D,
//
// with Q, K the normalised queries / keys (scale folded into Q) and S0 the request's [V, K] pool state. D is the
// record's delta, so the records hold (D, K, exp(g)) and the commit replays them.
//
// One wave per (request, value head, slice of 16 NTL value columns), 16 nodes on the 16 rows of the 16x16 MFMA
// accumulator (lane (g, c), element r: row 4 g + r, column c), each at its place():
//   - everything the wave reads is issued first: parents, gates, q / k rows, v, the pool slice;
//   - K K^T, K Q^T and Q Q^T on v_mfma_f32_16x16x32_bf16 from the raw bf16 rows (products exact, fp32 sums); the
//     squared norms are the diagonals, and the norms enter as per-row factors;
//   - per node (lane c): decay / beta, and by pointer jumping over the parent links the ancestor set (a 16-bit mask)
//     and the root-path log2-decay sum log2 G; the decay ratios are then hardware exp2 of log2 differences;
//   - L, L^T and W^T masked and scaled from K K^T and K Q^T;
//   - the triangular system by substitution over blocks of four nodes on v_mfma_f32_16x16x4f32, parents in front of
//     their children (rows given in another order are first ranked by depth);
//   - per 16-column tile, K S0^T and Q S0^T on the bf16 MFMA with the pool state split into exact bf16 terms
//     (1 for a bf16 pool, 2 for fp16, 3 for fp32), then rhs, D and O on the fp32 MFMA.
// Tile u of a wave covers the columns v0 + NTL c + u, so each lane ends with NTL adjacent columns of every row it
// holds: the records' deltas leave as 16 NTL-byte runs per lane.
// Work items are ordered so that the waves of one request's key head (its value heads and column slices) run on
// one XCD and share the q / k rows in its L2.

#include "gdn_walk.h"

namespace e4chunk {
int launch(const eagle4_records_args& a, hipStream_t s) __attribute__((visibility("hidden")));
}

namespace {

using namespace e4walk;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int NP = 16;  // nodes per request: the rows of one MFMA tile

E4_DEV f32x4_t mma_bf16(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                 0, 0, 0);
}

// X Y for 16 x 16 fp32 matrices in the accumulator layout, X passed transposed: block kb of the 16x16x4 MFMA
// contracts over k = 4 g + kb, for which a lane's A operand X[c][4 g + kb] is element kb of its X^T and its B operand
// Y[4 g + kb][c] element kb of its Y.
E4_DEV f32x4_t mm(f32x4_t xt, f32x4_t y, f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f}) {
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xt[kb], y[kb], acc, 0, 0, 0);
  return acc;
}

// The node at position p of a tile's 16 rows (and the position of a node: its own inverse): rows 4 g + b, element b of the
// lanes, hold nodes 4 b + g, so that what one MFMA contracts over (element b of the four lane groups) is a block of four
// consecutive nodes.
E4_DEV int place(int p) { return (p & ~15) | ((p & 3) << 2) | ((p >> 2) & 3); }

// A tile's triangular system by substitution over its blocks of four nodes: the blocks' own inverses, less I and
// transposed, (I + B)^-1 - I = B^2 - B - B^3 for the 4 x 4 blocks B of L (B^4 = 0), and with them D of (I + L) D = rhs - sub,
// LoT the rest of L transposed: element b of the lanes is block b, its right-hand side less what the blocks before it
// give. The product form of the whole inverse (powers up to L^8) cancels where keys along a path are alike and gates
// near one: the powers reach the thousands, and deltas of order one were off by 1e-3, by substitution 2e-6.
E4_DEV f32x4_t block_inverses(f32x4_t B, f32x4_t BT) {
  const f32x4_t B2T = mm(B, BT);
  return mm(B, -B2T, B2T - BT);
}
template <int N>
E4_DEV void solve_tiles(f32x4_t invT, f32x4_t LoT, const f32x4_t (&rhs)[N], f32x4_t (&sub)[N], f32x4_t (&D)[N]) {
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int u = 0; u < N; ++u) {  // column tiles: independent chains
      const float x = rhs[u][b] - sub[u][b];
      const f32x4_t z = __builtin_amdgcn_mfma_f32_16x16x4f32(invT[b], x, f32x4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      D[u][b] = x + z[b];
      if (b < 3) sub[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(LoT[b], D[u][b], sub[u], 0, 0, 0);
    }
}

// Loads whose width does not depend on a runtime dtype, so every dtype takes one code path and the compiler has no
// join at which to wait for loads in flight. A float input: the aligned 32-bit word holding element i (an allocation
// holds whole words) and the shift that brings the element to the low bits.
struct Word {
  uint32_t w;
  uint32_t sh;
};
E4_DEV Word word_of(const void* p, int64_t i, int dtype) {
  const int64_t byte = dtype == EAGLE4_F32 ? 4 * i : 2 * i;
  const uint32_t w = *reinterpret_cast<const uint32_t*>(static_cast<const char*>(p) + (byte & ~int64_t(3)));
  return {w, static_cast<uint32_t>(byte & 2) * 8u};
}
E4_DEV float widen_word(const Word& x, int dtype) {
  const uint32_t r = dtype == EAGLE4_F32 ? x.w : (x.w >> x.sh) & 0xffffu;
  return widen_raw(r, dtype);
}
// An integer table entry through its low 32 bits: int32, or int64 holding a value in int32 range (token offsets,
// slots, rows, parents).
E4_DEV int32_t entry(const eagle4_itab& t, int64_t i, int64_t j = 0) {
  const int64_t off = (i * t.s0 + j * t.s1) * (t.dtype == EAGLE4_I64 ? 8 : 4);
  return *reinterpret_cast<const int32_t*>(static_cast<const char*>(t.ptr) + off);
}

E4_DEV float lo_bf16(uint32_t w) { return __uint_as_float(w << 16); }
E4_DEV float hi_bf16(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
// Two fp32 values whose low 16 bits are zero (exact bf16 values) packed as bf16 elements 2 i, 2 i + 1.
E4_DEV uint32_t pack2(float x0, float x1) { return (__float_as_uint(x0) >> 16) | (__float_as_uint(x1) & 0xffff0000u); }
E4_DEV float trunc_bf16(float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); }

// The pool state as exact bf16 terms. A lane's slice of one tile and K block is 8 consecutive state elements (one
// row, k = 32 kb + 8 g ...); term 0 keeps the leading 8 significand bits (truncated), each further term those of what
// the earlier ones left, so the terms sum to the element exactly (fp16: 11 bits, 2 terms; fp32: 24 bits, 3 terms).
template <typename Tpool>
struct PoolTerms {
  static constexpr bool kF32 = sizeof(typename Tpool::storage) == 4;
  static constexpr int N = kF32 ? 3 : (Tpool::code == EAGLE4_F16 ? 2 : 1);
  static constexpr int WORDS = kF32 ? 2 : 1;  // uint4 per lane per (tile, K block)
  static E4_DEV void split(const uint4 (&raw)[WORDS], uint4 (&t)[N]) {
    if constexpr (N == 1) {
      t[0] = raw[0];
    } else {
      float x[8];
      if constexpr (kF32) {
        const uint32_t w[8] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w, raw[1].x, raw[1].y, raw[1].z, raw[1].w};
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = __uint_as_float(w[e]);
      } else {
        const uint32_t w[4] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[2 * e] = e4::f16_to_f32(static_cast<uint16_t>(w[e] & 0xffffu));
          x[2 * e + 1] = e4::f16_to_f32(static_cast<uint16_t>(w[e] >> 16));
        }
      }
      uint32_t p[N][4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float r0 = x[2 * e], r1 = x[2 * e + 1];
#pragma unroll
        for (int s = 0; s < N; ++s) {
          const float t0 = trunc_bf16(r0), t1 = trunc_bf16(r1);
          p[s][e] = pack2(t0, t1);
          r0 -= t0;  // exact: the bits below the kept ones
          r1 -= t1;
        }
      }
#pragma unroll
      for (int s = 0; s < N; ++s) t[s] = make_uint4(p[s][0], p[s][1], p[s][2], p[s][3]);
    }
  }
};

// NTL adjacent 16-bit elements (v inputs) as raw words.
template <int NTL>
struct Run16 {
  uint32_t w[(NTL + 1) / 2];
  E4_DEV void load(const uint16_t* p) {
    if constexpr (NTL == 4) {
      const uint2 x = *reinterpret_cast<const uint2*>(p);
      w[0] = x.x;
      w[1] = x.y;
    } else if constexpr (NTL == 2) {
      w[0] = *reinterpret_cast<const uint32_t*>(p);
    } else {
      w[0] = *p;
    }
  }
  E4_DEV float at(int u) const { return (u & 1) ? hi_bf16(w[u >> 1]) : lo_bf16(w[u >> 1]); }
};

template <int NTL>
E4_DEV void store_run_f32(float* p, const float (&x)[NTL]) {
  if constexpr (NTL == 4)
    *reinterpret_cast<float4*>(p) = make_float4(x[0], x[1], x[2], x[3]);
  else if constexpr (NTL == 2)
    *reinterpret_cast<float2*>(p) = make_float2(x[0], x[1]);
  else
    *p = x[0];
}

template <int NTL>
E4_DEV void store_run_out(void* base, int64_t i, int dtype, const float (&x)[NTL]) {
  if (dtype == EAGLE4_F32) {
    store_run_f32<NTL>(static_cast<float*>(base) + i, x);
    return;
  }
  uint16_t h[NTL];
#pragma unroll
  for (int u = 0; u < NTL; ++u) h[u] = dtype == EAGLE4_BF16 ? e4::f32_to_bf16(x[u]) : e4::f32_to_f16(x[u]);
  uint16_t* p = static_cast<uint16_t*>(base) + i;
  if constexpr (NTL == 4)
    *reinterpret_cast<uint2*>(p) = make_uint2(h[0] | (uint32_t(h[1]) << 16), h[2] | (uint32_t(h[3]) << 16));
  else if constexpr (NTL == 2)
    *reinterpret_cast<uint32_t*>(p) = h[0] | (uint32_t(h[1]) << 16);
  else
    *p = h[0];
}

template <int K, int NTL, typename Tpool>
__global__ __launch_bounds__(64) void gdn_chunk_kernel(const eagle4_records_args a, int slices, int per_xcd,
                                                        int total) {
  constexpr int KB = K / 32;
  using PT = PoolTerms<Tpool>;
  __shared__ float4 s_nd[NP];    // per node: ks, qs, beta, log G
  __shared__ uint32_t s_anc[NP];  // per node: strict ancestors
  __shared__ int s_id[NP];        // position -> row of the request

  // Work item: consecutive items share a key head (value heads of one group, then column slices); the hardware deals
  // workgroups to the 8 XCDs in turn, so item = (block % 8) * per_xcd + block / 8 gives each XCD one contiguous run.
  const int w = static_cast<int>(blockIdx.x % 8) * per_xcd + static_cast<int>(blockIdx.x / 8);
  if (w >= total) return;
  const int slice = w % slices, pair = w / slices;
  const int hv = pair % a.HV, n = pair / a.HV;
  const int ih = hv / (a.HV / a.H);
  const int lane = threadIdx.x, c = lane & 15, g = lane >> 4;

  // the request's table entries and the head's gate constants, all in flight together
  const int qs0 = entry(a.query_start_loc, n), qs1 = entry(a.query_start_loc, n + 1);
  const int rec_row = uni(entry(a.record_indices, n));
  const int idx = uni(entry(a.state_indices, n));
  const Word A_w = word_of(a.A_log, hv, a.A_log_dtype);
  const Word dt_w = word_of(a.dt_bias, hv, a.dt_bias_dtype);
  const int64_t bos = uni(qs0);
  int T = uni(qs1) - uni(qs0);
  T = T < a.width ? T : a.width;  // a tree has at most width (<= 16) rows
  if (T <= 0) return;

  // ---- every other load before the first wait -------------------------------------------------------------------
  const int par_raw = entry(a.parent, n, c < T ? c : T - 1);  // lane c is row c here
  Word ga, gb;
  uint4 qr[KB], kr[KB];
  Run16<NTL> vr[4];
  const int v0 = slice * 16 * NTL;
  auto load_rows = [&](auto&& row_of) {  // row_of(position): the request's row there, or one past the tree, where the
    auto row_at = [&](int p) {           // last row is read (finite values, masked below)
      const int row = row_of(p);
      return bos + (row < T ? row : T - 1);
    };
    const int64_t tok = row_at(c);
    ga = word_of(a.a, tok * a.stride_a + hv, a.gate_dtype);
    gb = word_of(a.b, tok * a.stride_b + hv, a.gate_dtype);
    const uint16_t* qp = static_cast<const uint16_t*>(a.q) + tok * a.stride_q + ih * K + 8 * g;
    const uint16_t* kp = static_cast<const uint16_t*>(a.k) + tok * a.stride_k + ih * K + 8 * g;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      qr[kb] = *reinterpret_cast<const uint4*>(qp + 32 * kb);
      kr[kb] = *reinterpret_cast<const uint4*>(kp + 32 * kb);
    }
    // v before the pool slice: loads complete in order, and the first tile needs v but only its own slice part
#pragma unroll
    for (int r = 0; r < 4; ++r)
      vr[r].load(static_cast<const uint16_t*>(a.v) + row_at(4 * g + r) * a.stride_v + static_cast<int64_t>(hv) * a.V + v0 +
                 NTL * c);
  };
  load_rows(place);
  // The pool slice (rows v0 .. v0 + 16 NTL of the request's slot) through a buffer resource whose range is the slice,
  // or empty for a negative slot index: its loads then return zeros, the zero initial state (:341-345), with no
  // branch around them.
  using PS = typename Tpool::storage;
  constexpr int kSliceBytes = 16 * NTL * K * static_cast<int>(sizeof(PS));
  const char* slot = static_cast<const char*>(a.state) +
                     ((idx >= 0 ? static_cast<int64_t>(idx) * a.stride_state : 0) +
                      (static_cast<int64_t>(hv) * a.V + v0) * K) * static_cast<int64_t>(sizeof(PS));
  const __amdgpu_buffer_rsrc_t srsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(slot), 0, idx >= 0 ? kSliceBytes : 0, 0x00020000);
  uint4 sraw[NTL][KB][PT::WORDS];
#pragma unroll
  for (int u = 0; u < NTL; ++u)
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int q = 0; q < PT::WORDS; ++q) {
        const int off = ((NTL * c + u) * K + 32 * kb + 8 * g) * static_cast<int>(sizeof(PS)) + 16 * q;
        sraw[u][kb][q] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(srsrc, off, 0, 0));
      }
  // keep the scheduler from sinking these loads below the per-node math that waits for the q / k rows
  __builtin_amdgcn_sched_barrier(0);

  // ---- the order of the nodes: parents first -------------------------------------------------------------------------
  // a parent outside the tree (or the node itself) makes the node a root
  const int par_row = c > 0 && c < T && par_raw >= 0 && par_raw < T && par_raw != c ? par_raw : -1;
  int row_c = place(c), par;  // from here on lane c is the node at position c: its row, its parent's position
  if (__ballot(par_row > c) == 0) {
    const int up = __shfl(par_row, row_c, 16);
    par = up >= 0 ? place(up) : -1;
  } else {  // rank the rows by (depth, row)
    int depth = 0;
    for (int it = 0, x = par_row; it < T; ++it) {  // one step up for every lane; all lanes take part in the shuffle
      const int up = __shfl(par_row, x >= 0 ? x : 0, 16);
      if (x >= 0) {
        ++depth;
        x = up;
      }
    }
    const int key = c < T ? depth * 16 + c : 16 * 32 + c;
    int rank = 0;
    for (int j = 0; j < 16; ++j) rank += readlane(key, j) < key ? 1 : 0;
    s_id[place(rank)] = c;
    __syncthreads();
    row_c = s_id[c];
    const int up = __shfl(par_row, row_c, 16), up_rank = __shfl(rank, up >= 0 ? up : 0, 16);
    par = up >= 0 ? place(up_rank) : -1;
    load_rows([&](int p) { return s_id[p]; });
    settle_loads();  // else the waits after the join would take the common path's first loads for its last
  }
  const bool in = place(c) < T;  // a rank past the tree's is none of its rows

  // ---- node x node products; their diagonals are the squared norms ---------------------------------------------------
  f32x4_t KK = {0.f, 0.f, 0.f, 0.f}, KQ = {0.f, 0.f, 0.f, 0.f}, QQ = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    KK = mma_bf16(kr[kb], kr[kb], KK);  // KK[i][j] = k_i . k_j
    KQ = mma_bf16(kr[kb], qr[kb], KQ);  // KQ[i][j] = k_i . q_j
    QQ = mma_bf16(qr[kb], qr[kb], QQ);  // QQ[i][j] = q_i . q_j
  }

  // ---- per node (lane c): gates, ancestors, root-path log decay -----------------------------------------------------
  const float A = -expf(widen_word(A_w, a.A_log_dtype));
  const float dt_bias = widen_word(dt_w, a.dt_bias_dtype);
  const uint32_t ga_raw = a.gate_dtype == EAGLE4_F32 ? ga.w : (ga.w >> ga.sh) & 0xffffu;
  const uint32_t gb_raw = a.gate_dtype == EAGLE4_F32 ? gb.w : (gb.w >> gb.sh) & 0xffffu;
  const float2 gt = gate_of(ga_raw, gb_raw, a.gate_dtype, 1.0f, 20.0f, A, dt_bias);
  const float decay = in ? gt.x : 1.0f, beta = in ? gt.y : 0.0f;  // past the tree: exp(g) 1, beta 0 (:316-317)
  // pointer jumping: after round j, anc holds the ancestors at distance 1 .. 2^j, lsum the log2 decays of the node and
  // its ancestors at distance < 2^j, jmp the ancestor at distance 2^j (-1 past the root); depth < 16 needs 4 rounds.
  // Decay ratios are then powers of two of log2 differences (the hardware exp2 / log2, ~1 ulp).
  uint32_t anc = par >= 0 ? 1u << par : 0u;
  int jmp = par;
  float lsum = __builtin_amdgcn_logf(fmaxf(decay, 1e-30f));
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int src = jmp >= 0 ? jmp : c;
    const uint32_t anc_j = static_cast<uint32_t>(__shfl(static_cast<int>(anc), src, 16));
    const int jmp_j = __shfl(jmp, src, 16);
    const float l_j = __shfl(lsum, src, 16);
    if (jmp >= 0) {
      anc |= anc_j;
      lsum += l_j;
      jmp = jmp_j;
    }
  }
  const float logG = lsum;  // log2 G
  // node c's squared norms sit on the diagonals at lane (c / 4, c), element c % 4; that lane publishes the node
  const int rc = c & 3;
  const float kk = rc == 0 ? KK[0] : rc == 1 ? KK[1] : rc == 2 ? KK[2] : KK[3];
  const float qq = rc == 0 ? QQ[0] : rc == 1 ? QQ[1] : rc == 2 ? QQ[2] : QQ[3];
  if (g == (c >> 2)) {
    s_nd[c] = make_float4(1.0f / sqrtf(kk + 1e-6f), a.scale / sqrtf(qq + 1e-6f), beta, logG);  // (:147-150)
    s_anc[c] = anc;
    s_id[c] = row_c;
  }
  __syncthreads();
  const float ks = s_nd[c].x, qs = s_nd[c].y;
  // the record's key and decay (once per node and value head) leave now, ahead of the matrix work
  float* rec = a.records + static_cast<int64_t>(rec_row) * a.stride_records_row;
  if (slice == 0 && rec_row >= 0 && in) {
    float* p = rec + (static_cast<int64_t>(row_c) * a.HV + hv) * a.rec + a.V;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const uint4 x = kr[kb];
      float4* d = reinterpret_cast<float4*>(p + 32 * kb + 8 * g);
      d[0] = make_float4(lo_bf16(x.x) * ks, hi_bf16(x.x) * ks, lo_bf16(x.y) * ks, hi_bf16(x.y) * ks);
      d[1] = make_float4(lo_bf16(x.z) * ks, hi_bf16(x.z) * ks, lo_bf16(x.w) * ks, hi_bf16(x.w) * ks);
    }
    if (g == 0) p[K] = decay;
  }

  // ---- L, L^T, W^T -------------------------------------------------------------------------------------------------
  float4 nd[4];
  float Gr[4];
  f32x4_t B, BT, LoT, WT;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 4 * g + r;
    nd[r] = s_nd[i];
    const uint32_t anc_i = s_anc[i];
    Gr[r] = __builtin_amdgcn_exp2f(nd[r].w);
    const bool c_above_i = (anc_i >> c) & 1u;  // c a strict ancestor of i
    const bool i_above_c = (anc >> i) & 1u;    // i a strict ancestor of c
    const float kk_n = nd[r].x * ks * KK[r];
    // L[i][c] = beta_i G_i / G_c k^_i . k^_c on strict ancestors c of i
    const float l = c_above_i ? nd[r].z * __builtin_amdgcn_exp2f(nd[r].w - logG) * kk_n : 0.f;
    // L^T[i][c] = L[c][i];  W^T[i][c] = W[c][i] = G_c / G_i q^_c . k^_i on ancestors-or-self i of c
    const float ratio = i_above_c || i == c ? __builtin_amdgcn_exp2f(logG - nd[r].w) : 0.f;
    const float lt = i_above_c ? beta * ratio * kk_n : 0.f;
    const bool own = (c & 3) == r;  // nodes i and c in one block of four
    B[r] = own ? l : 0.f;
    BT[r] = own ? lt : 0.f;
    LoT[r] = own ? 0.f : lt;
    WT[r] = ratio * (qs * nd[r].x * KQ[r]);
  }
  const f32x4_t invT = block_inverses(B, BT);

  // ---- per 16-column tile: K S0^T, Q S0^T, rhs, D, O = G Q S0^T + W D ------------------------------------
  f32x4_t rhs[NTL], D[NTL], O[NTL], sub[NTL];
#pragma unroll
  for (int u = 0; u < NTL; ++u) {
    f32x4_t KS = {0.f, 0.f, 0.f, 0.f}, QS = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      uint4 st[PT::N];
      PT::split(sraw[u][kb], st);
#pragma unroll
      for (int s = 0; s < PT::N; ++s) {
        KS = mma_bf16(kr[kb], st[s], KS);
        QS = mma_bf16(qr[kb], st[s], QS);
      }
    }
    sub[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      rhs[u][r] = 4 * r + g < T ? nd[r].z * (vr[r].at(u) - Gr[r] * (nd[r].x * KS[r])) : 0.f;
      O[u][r] = Gr[r] * (nd[r].y * QS[r]);
    }
  }
  solve_tiles<NTL>(invT, LoT, rhs, sub, D);
#pragma unroll
  for (int u = 0; u < NTL; ++u) O[u] += mm(WT, D[u]);

  // ---- stores --------------------------------------------------------------------------------------------------------
  const int64_t col = static_cast<int64_t>(hv) * a.V + v0 + NTL * c;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (4 * r + g < T) {
      const int i = s_id[4 * g + r];
      float o[NTL], d[NTL];
#pragma unroll
      for (int u = 0; u < NTL; ++u) {
        o[u] = O[u][r];
        d[u] = D[u][r];
      }
      store_run_out<NTL>(a.out, (bos + i) * a.stride_o + col, a.out_dtype, o);
      if (rec_row >= 0) store_run_f32<NTL>(rec + (static_cast<int64_t>(i) * a.HV + hv) * a.rec + v0 + NTL * c, d);
    }
  }
}

template <int K, int NTL>
int launch_pool(const eagle4_records_args& a, hipStream_t s) {
  const int slices = a.V / (16 * NTL);
  const int64_t total = static_cast<int64_t>(a.N) * a.HV * slices;
  if (total > (int64_t(1) << 30)) return EAGLE4_NOT_COVERED;
  const int per_xcd = static_cast<int>((total + 7) / 8);
  const dim3 grid(8 * per_xcd);
  const int t = static_cast<int>(total);
  if (a.state_dtype == EAGLE4_BF16)
    gdn_chunk_kernel<K, NTL, e4::Bf16><<<grid, 64, 0, s>>>(a, slices, per_xcd, t);
  else if (a.state_dtype == EAGLE4_F16)
    gdn_chunk_kernel<K, NTL, e4::F16><<<grid, 64, 0, s>>>(a, slices, per_xcd, t);
  else if constexpr (NTL < 4)  // four tiles of an fp32 slice would not fit the registers
    if (a.state_dtype == EAGLE4_F32)
      gdn_chunk_kernel<K, NTL, e4::F32><<<grid, 64, 0, s>>>(a, slices, per_xcd, t);
    else
      return EAGLE4_NOT_COVERED;
  else
    return EAGLE4_NOT_COVERED;
  return E4_LAUNCH_STATUS();
}

template <int K>
int launch_k(const eagle4_records_args& a, hipStream_t s) {
  // columns per wave: more columns per wave once there are enough waves to keep HBM busy (measured at 16 / 48 heads,
  // K = V = 128: 1 tile per wave at 1 request, 2 at 4, 4 at 16 and 32)
  const int64_t pairs = static_cast<int64_t>(a.N) * a.HV;
  const bool fp32_pool = a.state_dtype == EAGLE4_F32;
  if constexpr (K <= 128)
    if (!fp32_pool && a.V % 64 == 0 && pairs * (a.V / 64) >= 1024) return launch_pool<K, 4>(a, s);
  if (a.V % 32 == 0 && pairs * (a.V / 32) >= 512) return launch_pool<K, 2>(a, s);
  return launch_pool<K, 1>(a, s);
}

// ---- trees of 17 to 64 nodes ---------------------------------------------------------------------------------------
// The same closed form, blocked by tiles of 16 nodes: with every parent in front of its children L is block lower
// triangular, so the tiles are solved in order,
//   D_I = (I + L_II)^-1 (rhs_I - sum_{J<I} L_IJ D_J),   O_I = diag(G) Q_I S0^T + sum_{J<=I} W_IJ D_J,
// each 16 x 16 block on the MFMA as above, the blocks of tile I built when it is solved (they are used at once by the
// wave's NTL column tiles, nothing is kept but D). One wave per (request, value head, 16 NTL columns). Rows given in
// another order are first ranked by depth. Bound by one wave's latency: at K 128 and three or four tiles a wave holds 250
// to 300 registers, so one or two fit a SIMD, and the tiles are a serial chain. Of a wave's cycles at 8 requests of 20 - 40
// nodes, 32 heads (at 32 of 64 nodes, 48 heads) the MFMA is busy for 19 % (26), the VALU issues for 25 % (29), and 34 %
// (26) are waits for loads and LDS. The walk that it replaces steps through the nodes one by one, each a chain of two
// lane sums. K = V = 128, fp32 pool, kernel against the walk: 1 request of 24 nodes, 16 heads 33.4 -> 8.6 us; 8 of 40
// nodes, 48 heads 318 -> 29 us; 32 of 64 nodes, 48 heads 2108 -> 141 us.
//   - Decay ratios are exp2 of differences of root-path sums of log2 decays; the sums are fp64, so what two nodes share
//     cancels exactly and the ratio's error is that of the path between them, whatever the root path's length.
//   - A value that is not finite stays on its node and the node's descendants, as in a walk: products with zeros would
//     spread it over the tile, so it is taken out of the right-hand sides (and a node with such a key or gate out of
//     the products), remembered per column, and put back where the outputs of that path are stored: NaN, as in the walk,
//     whose states then hold infinities of both signs; the delta of an infinite value itself stays infinite.
template <int K, int NTL, int NTILE, typename Tpool>
__global__ __launch_bounds__(64) void gdn_chunk_wide_kernel(const eagle4_records_args a, int slices, int per_xcd,
                                                             int total) {
  constexpr int KB = K / 32;
  constexpr int NN = 16 * NTILE;
  constexpr int ROUNDS = NN <= 32 ? 5 : 6;  // pointer jumping: depth < 2^ROUNDS
  using PT = PoolTerms<Tpool>;
  __shared__ float4 s_nd[64];     // per node: ks, qs, beta, G
  __shared__ double s_lg[64];     // per node: log2 G
  __shared__ uint64_t s_anc[64];  // per node: strict ancestors
  __shared__ float2 s_nrm[64];    // per node: |k|^2, |q|^2
  __shared__ int s_id[64];        // position -> row of the request
  __shared__ float s_raw[NTL][4][64];  // a tile's right-hand sides that are not finite, each lane its own

  const int w = static_cast<int>(blockIdx.x % 8) * per_xcd + static_cast<int>(blockIdx.x / 8);
  if (w >= total) return;
  const int slice = w % slices, pair = w / slices;
  const int hv = pair % a.HV, n = pair / a.HV;
  const int ih = hv / (a.HV / a.H);
  const int lane = threadIdx.x, c = lane & 15, g = lane >> 4;

  const int qs0 = entry(a.query_start_loc, n), qs1 = entry(a.query_start_loc, n + 1);
  const int rec_row = uni(entry(a.record_indices, n));
  const int idx = uni(entry(a.state_indices, n));
  const Word A_w = word_of(a.A_log, hv, a.A_log_dtype);
  const Word dt_w = word_of(a.dt_bias, hv, a.dt_bias_dtype);
  const int64_t bos = uni(qs0);
  int T = uni(qs1) - uni(qs0);
  T = T < a.width ? T : a.width;  // a tree has at most width (<= 16 NTILE) rows
  if (T <= 0) return;

  // ---- every load before the first wait; rows past the tree read its last row (masked below) ------------------------
  const int par_raw = entry(a.parent, n, lane < T ? lane : T - 1);
  const int node = place(lane);  // the node at position `lane`
  uint4 qr[NTILE][KB], kr[NTILE][KB];
  Run16<NTL> vr[NTILE][4];
  Word ga, gb;
  const int v0 = slice * 16 * NTL;
  auto load_rows = [&](auto&& row_of) {  // row_of(position): the request's row there, or one past the tree
    auto row_at = [&](int p) {
      const int row = row_of(p);
      return bos + (row < T ? row : T - 1);
    };
    const int64_t tl = row_at(lane);
    ga = word_of(a.a, tl * a.stride_a + hv, a.gate_dtype);
    gb = word_of(a.b, tl * a.stride_b + hv, a.gate_dtype);
#pragma unroll
    for (int I = 0; I < NTILE; ++I) {
      const int64_t tok = row_at(16 * I + c);
      const uint16_t* qp = static_cast<const uint16_t*>(a.q) + tok * a.stride_q + ih * K + 8 * g;
      const uint16_t* kp = static_cast<const uint16_t*>(a.k) + tok * a.stride_k + ih * K + 8 * g;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        qr[I][kb] = *reinterpret_cast<const uint4*>(qp + 32 * kb);
        kr[I][kb] = *reinterpret_cast<const uint4*>(kp + 32 * kb);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t ti = row_at(16 * I + 4 * g + r);
        vr[I][r].load(static_cast<const uint16_t*>(a.v) + ti * a.stride_v + static_cast<int64_t>(hv) * a.V + v0 + NTL * c);
      }
    }
  };
  load_rows(place);
  using PS = typename Tpool::storage;
  constexpr int kSliceBytes = 16 * NTL * K * static_cast<int>(sizeof(PS));
  const char* slot = static_cast<const char*>(a.state) +
                     ((idx >= 0 ? static_cast<int64_t>(idx) * a.stride_state : 0) +
                      (static_cast<int64_t>(hv) * a.V + v0) * K) * static_cast<int64_t>(sizeof(PS));
  const __amdgpu_buffer_rsrc_t srsrc =  // empty for a negative slot: zeros
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(slot), 0, idx >= 0 ? kSliceBytes : 0, 0x00020000);
  uint4 sraw[NTL][KB][PT::WORDS];
#pragma unroll
  for (int u = 0; u < NTL; ++u)
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int q = 0; q < PT::WORDS; ++q) {
        const int off = ((NTL * c + u) * K + 32 * kb + 8 * g) * static_cast<int>(sizeof(PS)) + 16 * q;
        sraw[u][kb][q] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(srsrc, off, 0, 0));
      }
  __builtin_amdgcn_sched_barrier(0);

  // ---- the order of the nodes: parents first -------------------------------------------------------------------------
  // lane r is row r here; a parent outside the tree (or the node itself) makes the node a root
  const int par_row = lane > 0 && lane < T && par_raw >= 0 && par_raw < T && par_raw != lane ? par_raw : -1;
  const bool reordered = __ballot(par_row > lane) != 0;
  int rank = lane;
  if (reordered) {  // rank the rows by (depth, row)
    int depth = 0;
    for (int it = 0, x = par_row; it < T; ++it) {  // one step up for every lane; all lanes take part in the shuffle
      const int up = __shfl(par_row, x >= 0 ? x : 0);
      if (x >= 0) {
        ++depth;
        x = up;
      }
    }
    const int key = lane < T ? depth * 64 + lane : 64 * 128 + lane;
    rank = 0;
    for (int j = 0; j < 64; ++j) rank += readlane(key, j) < key ? 1 : 0;
  }
  s_id[place(rank)] = lane;
  __syncthreads();
  // from here on lane p is the node at position p
  int par;
  {
    const int up = __shfl(par_row, s_id[lane]);
    const int up_rank = __shfl(rank, up >= 0 ? up : 0);
    par = up >= 0 ? place(up_rank) : -1;
  }
  if (reordered) load_rows([&](int p) { return s_id[p]; });

  // ---- per node (lane p): gates, ancestors, root-path log decay; squared norms from the tiles' diagonals --------------
  const float A = -expf(widen_word(A_w, a.A_log_dtype));
  const float dt_bias = widen_word(dt_w, a.dt_bias_dtype);
#pragma unroll
  for (int I = 0; I < NTILE; ++I) {
    f32x4_t KK = {0.f, 0.f, 0.f, 0.f}, QQ = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      KK = mma_bf16(kr[I][kb], kr[I][kb], KK);
      QQ = mma_bf16(qr[I][kb], qr[I][kb], QQ);
    }
    const int rc = c & 3;
    const float kk = rc == 0 ? KK[0] : rc == 1 ? KK[1] : rc == 2 ? KK[2] : KK[3];
    const float qq = rc == 0 ? QQ[0] : rc == 1 ? QQ[1] : rc == 2 ? QQ[2] : QQ[3];
    if (g == (c >> 2)) s_nrm[16 * I + c] = make_float2(kk, qq);
  }
  const float2 gt = gate_of(a.gate_dtype == EAGLE4_F32 ? ga.w : (ga.w >> ga.sh) & 0xffffu,
                            a.gate_dtype == EAGLE4_F32 ? gb.w : (gb.w >> gb.sh) & 0xffffu, a.gate_dtype, 1.0f, 20.0f,
                            A, dt_bias);
  const float x_dt = widen_word(ga, a.gate_dtype) + dt_bias;
  const float gl = A * (x_dt <= 20.0f ? logf(1.0f + expf(x_dt)) : x_dt);  // gate_of's log decay
  uint64_t anc = par >= 0 ? 1ull << par : 0ull;
  int jmp = par;
  double lsum = node < T ? fmax(static_cast<double>(gl) * 1.4426950408889634, -1048576.0) : 0.0;
#pragma unroll
  for (int it = 0; it < ROUNDS; ++it) {
    const int src = jmp >= 0 ? jmp : lane;
    const uint32_t lo = static_cast<uint32_t>(__shfl(static_cast<int>(anc & 0xffffffffu), src));
    const uint32_t hi = NN > 32 ? static_cast<uint32_t>(__shfl(static_cast<int>(anc >> 32), src)) : 0u;
    const int jmp_j = __shfl(jmp, src);
    const double l_j = __shfl(lsum, src);
    if (jmp >= 0) {
      anc |= (static_cast<uint64_t>(hi) << 32) | lo;
      lsum += l_j;
      jmp = jmp_j;
    }
  }
  __syncthreads();
  const float2 nrm = s_nrm[lane < NN ? lane : 0];
  const float ks_l = 1.0f / sqrtf(nrm.x + 1e-6f);
  const bool gates = fabsf(gt.x) <= 3.4e38f && fabsf(gt.y) <= 3.4e38f;
  const uint64_t inf_k = __ballot(node < T && !(nrm.x <= 3.4e38f));
  const uint64_t inf_q = __ballot(node < T && !(nrm.y <= 3.4e38f));
  uint64_t bad = inf_k | __ballot(node < T && !gates);  // nodes whose key or gate is not finite
  const bool use = node < T && gates;
  s_nd[lane] = make_float4(use && ((bad >> lane) & 1) == 0 ? ks_l : 0.f, a.scale / sqrtf(nrm.y + 1e-6f), use ? gt.y : 0.f,
                           __builtin_amdgcn_exp2f(static_cast<float>(lsum)));
  s_lg[lane] = lsum;
  s_anc[lane] = anc;
  __syncthreads();
  // the records' keys and decays (once per node and value head) leave ahead of the matrix work
  float* rec = a.records + static_cast<int64_t>(rec_row) * a.stride_records_row;
  if (slice == 0 && rec_row >= 0) {
#pragma unroll
    for (int I = 0; I < NTILE; ++I) {
      const int p = 16 * I + c;
      if (place(p) < T) {
        float* d0 = rec + (static_cast<int64_t>(s_id[p]) * a.HV + hv) * a.rec + a.V;
        const float ks = 1.0f / sqrtf(s_nrm[p].x + 1e-6f);
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          const uint4 x = kr[I][kb];
          float4* d = reinterpret_cast<float4*>(d0 + 32 * kb + 8 * g);
          d[0] = make_float4(lo_bf16(x.x) * ks, hi_bf16(x.x) * ks, lo_bf16(x.y) * ks, hi_bf16(x.y) * ks);
          d[1] = make_float4(lo_bf16(x.z) * ks, hi_bf16(x.z) * ks, lo_bf16(x.w) * ks, hi_bf16(x.w) * ks);
        }
      }
    }
    if (node < T) rec[(static_cast<int64_t>(s_id[lane]) * a.HV + hv) * a.rec + a.V + K] = gt.x;
  }
  if (bad != 0) {
#pragma unroll
    for (int I = 0; I < NTILE; ++I)
      if ((bad >> (16 * I + c)) & 1) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) kr[I][kb] = make_uint4(0u, 0u, 0u, 0u);
      }
  }

  // ---- K S0^T and Q S0^T of every tile -------------------------------------------------------------------------------
  f32x4_t KS[NTILE][NTL], QS[NTILE][NTL];
#pragma unroll
  for (int I = 0; I < NTILE; ++I)
#pragma unroll
    for (int u = 0; u < NTL; ++u) {
      KS[I][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      QS[I][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
  for (int u = 0; u < NTL; ++u)
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      uint4 st[PT::N];
      PT::split(sraw[u][kb], st);
#pragma unroll
      for (int s = 0; s < PT::N; ++s)
#pragma unroll
        for (int I = 0; I < NTILE; ++I) {
          KS[I][u] = mma_bf16(kr[I][kb], st[s], KS[I][u]);
          QS[I][u] = mma_bf16(qr[I][kb], st[s], QS[I][u]);
        }
    }

  // ---- the tiles in order ---------------------------------------------------------------------------------------------
  f32x4_t D[NTILE][NTL];
  uint64_t lost[NTL];  // column v0 + NTL c + u: the nodes whose right-hand side is not finite
#pragma unroll
  for (int u = 0; u < NTL; ++u) lost[u] = 0;
  // A row of finite elements whose squared norm overflows is a zero row once normalised (1 / inf): the key is out of the
  // products already, and its node is not bad. One that holds an infinity or a NaN stays what it is.
  uint64_t zero_q = 0;
  bool any_lost = (bad | inf_q) != 0;
  if (any_lost) {
    auto rows_with_inf = [&](const void* x, int64_t stride) -> uint64_t {  // read again, a lane its own row
      const uint16_t* p = static_cast<const uint16_t*>(x) + (bos + (node < T ? s_id[lane] : 0)) * stride + ih * K;
      bool hit = false;
#pragma unroll 1
      for (int e = 0; e < K; ++e) hit |= (p[e] & 0x7f80u) == 0x7f80u;
      return __ballot(hit);
    };
    bad &= ~inf_k | rows_with_inf(a.k, a.stride_k) | __ballot(!use);
    zero_q = inf_q & ~rows_with_inf(a.q, a.stride_q);
  }
#pragma unroll
  for (int I = 0; I < NTILE; ++I) {
    if (16 * I >= T) break;
    const float4 ci = s_nd[16 * I + c];  // the node of this lane's column
    const double lg_c = s_lg[16 * I + c];
    const uint64_t anc_c = s_anc[16 * I + c];
    f32x4_t sub[NTL], out[NTL], rhs[NTL];
#pragma unroll
    for (int u = 0; u < NTL; ++u) {
      sub[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      out[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int J = 0; J < I; ++J) {
      f32x4_t KK = {0.f, 0.f, 0.f, 0.f}, KQ = {0.f, 0.f, 0.f, 0.f}, LT, WT;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        KK = mma_bf16(kr[J][kb], kr[I][kb], KK);
        KQ = mma_bf16(kr[J][kb], qr[I][kb], KQ);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = 16 * J + 4 * g + r;
        const float ks_j = s_nd[j].x;
        const float ratio = __builtin_amdgcn_exp2f(static_cast<float>(lg_c - s_lg[j]));
        const bool above = (anc_c >> j) & 1;
        LT[r] = above ? ci.z * ratio * (ks_j * ci.x * KK[r]) : 0.f;  // L^T: L[c][j]
        WT[r] = above ? ratio * (ci.y * ks_j * KQ[r]) : 0.f;         // W^T
      }
#pragma unroll
      for (int u = 0; u < NTL; ++u) {
        sub[u] = mm(LT, D[J][u], sub[u]);
        out[u] = mm(WT, D[J][u], out[u]);
      }
    }
    f32x4_t KK = {0.f, 0.f, 0.f, 0.f}, KQ = {0.f, 0.f, 0.f, 0.f}, B, BT, LoT, WT;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      KK = mma_bf16(kr[I][kb], kr[I][kb], KK);
      KQ = mma_bf16(kr[I][kb], qr[I][kb], KQ);
    }
    float4 nd[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * g + r, ni = 16 * I + i;
      nd[r] = s_nd[ni];
      const double lg_i = s_lg[ni];
      const bool c_above_i = (s_anc[ni] >> (16 * I + c)) & 1, i_above_c = (anc_c >> ni) & 1;
      const float kk_n = nd[r].x * ci.x * KK[r];
      const float ratio = i_above_c || i == c ? __builtin_amdgcn_exp2f(static_cast<float>(lg_c - lg_i)) : 0.f;
      const float l = c_above_i ? nd[r].z * __builtin_amdgcn_exp2f(static_cast<float>(lg_i - lg_c)) * kk_n : 0.f;
      const float lt = i_above_c ? ci.z * ratio * kk_n : 0.f;
      const bool own = (c & 3) == r;  // nodes i and c in one block of four
      B[r] = own ? l : 0.f;
      BT[r] = own ? lt : 0.f;
      LoT[r] = own ? 0.f : lt;
      WT[r] = i_above_c || i == c ? ratio * (ci.y * nd[r].x * KQ[r]) : 0.f;
    }
    const f32x4_t invT = block_inverses(B, BT);
#pragma unroll
    for (int u = 0; u < NTL; ++u) {
      bool off = false;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        rhs[u][r] = 16 * I + 4 * r + g < T ? nd[r].z * (vr[I][r].at(u) - nd[r].w * (nd[r].x * KS[I][u][r])) : 0.f;
        off |= !(fabsf(rhs[u][r] - sub[u][r]) <= 3.4e38f);
      }
      if (__ballot(off) != 0) {  // take what is not finite out of the products, remember where it was
        uint32_t m = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (!(fabsf(rhs[u][r] - sub[u][r]) <= 3.4e38f)) {
            m |= 1u << (4 * g + r);
            s_raw[u][r][lane] = rhs[u][r] - sub[u][r];
            rhs[u][r] = sub[u][r] = 0.f;
          }
        m |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), 16));
        m |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), 32));
        lost[u] |= static_cast<uint64_t>(m) << (16 * I);
        any_lost = true;
      }
    }
    solve_tiles<NTL>(invT, LoT, rhs, sub, D[I]);
#pragma unroll
    for (int u = 0; u < NTL; ++u) out[u] = mm(WT, D[I][u], out[u]);
    // ---- the tile's outputs and deltas ----
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int p = 16 * I + 4 * g + r;
      if (place(p) >= T) continue;
      float o[NTL], d[NTL];
#pragma unroll
      for (int u = 0; u < NTL; ++u) {
        o[u] = nd[r].w * (nd[r].y * QS[I][u][r]) + out[u][r];
        d[u] = D[I][u][r];
      }
      if (any_lost) {
        const uint64_t above = s_anc[p], self = 1ull << p;
#pragma unroll
        for (int u = 0; u < NTL; ++u)
          if (((above | self) & (lost[u] | bad)) == 0) {
            if ((zero_q & self) != 0) o[u] = 0.f;
          } else {
            o[u] = __builtin_nanf("");
            const float own = s_raw[u][r][lane];  // an infinite value's own delta
            d[u] = (lost[u] & self) != 0 && (above & (lost[u] | bad)) == 0 ? own : __builtin_nanf("");
          }
      }
      const int row = s_id[p];
      const int64_t col = static_cast<int64_t>(hv) * a.V + v0 + NTL * c;
      store_run_out<NTL>(a.out, (bos + row) * a.stride_o + col, a.out_dtype, o);
      if (rec_row >= 0) store_run_f32<NTL>(rec + (static_cast<int64_t>(row) * a.HV + hv) * a.rec + v0 + NTL * c, d);
    }
  }
}

template <int K, int NTL, int NTILE>
int launch_wide_pool(const eagle4_records_args& a, hipStream_t s) {
  const int slices = a.V / (16 * NTL);
  const int64_t total = static_cast<int64_t>(a.N) * a.HV * slices;
  if (total > (int64_t(1) << 30)) return EAGLE4_NOT_COVERED;
  const int per_xcd = static_cast<int>((total + 7) / 8);
  const int t = static_cast<int>(total);
  if (a.state_dtype == EAGLE4_BF16)
    gdn_chunk_wide_kernel<K, NTL, NTILE, e4::Bf16><<<8 * per_xcd, 64, 0, s>>>(a, slices, per_xcd, t);
  else if (a.state_dtype == EAGLE4_F16)
    gdn_chunk_wide_kernel<K, NTL, NTILE, e4::F16><<<8 * per_xcd, 64, 0, s>>>(a, slices, per_xcd, t);
  else if (a.state_dtype == EAGLE4_F32)
    gdn_chunk_wide_kernel<K, NTL, NTILE, e4::F32><<<8 * per_xcd, 64, 0, s>>>(a, slices, per_xcd, t);
  else
    return EAGLE4_NOT_COVERED;
  return E4_LAUNCH_STATUS();
}

// Two column tiles per wave halve the work on the node blocks that the waves of a head repeat, one gives twice the
// waves: from 512 waves of two on, two are faster (32 requests of 64 nodes, 48 heads 157 against 205 us; 8 of 24 nodes,
// 16 heads: 512 waves, 12.9 against 12.2, of 64 nodes 24.8 against 24.7; 2 of 64 nodes, 48 heads: 384 waves, 23.7
// against 21.3).
template <int K, int NTILE>
int launch_wide(const eagle4_records_args& a, hipStream_t s) {
  const int64_t pairs = static_cast<int64_t>(a.N) * a.HV;
  if (a.V % 32 == 0 && pairs * (a.V / 32) >= 512) return launch_wide_pool<K, 2, NTILE>(a, s);
  return launch_wide_pool<K, 1, NTILE>(a, s);
}

template <int K>
int launch_wide_k(const eagle4_records_args& a, hipStream_t s) {
  if (a.width <= 32) return launch_wide<K, 2>(a, s);
  if (a.width <= 48) return launch_wide<K, 3>(a, s);
  return launch_wide<K, 4>(a, s);
}

}  // namespace

namespace e4chunk {

// The chunk form on the matrix cores when it covers the call: no path table, bf16 inputs, a key dim of 32 .. 256 for
// trees of <= 16 nodes and of 32 .. 128 up to 64 nodes (four tiles of 256-wide rows would not fit the registers), value
// dim a multiple of 16, 16-byte aligned rows. Returns EAGLE4_NOT_COVERED (nothing launched) otherwise.
int launch(const eagle4_records_args& a, hipStream_t s) {
  const auto al = [](const void* p, int64_t bytes) { return reinterpret_cast<uintptr_t>(p) % bytes == 0; };
  if (a.path_replay || a.width > 64 || a.in_dtype != EAGLE4_BF16 || a.V % 16 || a.stride_q % 8 || a.stride_k % 8 ||
      a.stride_v % 4 || a.stride_o % 4 || a.rec % 4 || a.stride_records_row % 4 || !al(a.q, 16) || !al(a.k, 16) ||
      !al(a.v, 8) || !al(a.out, 16) || !al(a.records, 16) || !al(a.state, 16) || a.stride_state % 8)
    return EAGLE4_NOT_COVERED;
  if (a.width > NP) {
    switch (a.K) {
      case 32: return launch_wide_k<32>(a, s);
      case 64: return launch_wide_k<64>(a, s);
      case 128: return launch_wide_k<128>(a, s);
      default: return EAGLE4_NOT_COVERED;
    }
  }
  switch (a.K) {
    case 32: return launch_k<32>(a, s);
    case 64: return launch_k<64>(a, s);
    case 128: return launch_k<128>(a, s);
    case 256: return launch_k<256>(a, s);
    default: return EAGLE4_NOT_COVERED;
  }
}

}  // namespace e4chunk
