// Kernels of the three-body (CHGNet/MatRIS-style) model: the bond envelope of the line graph,
// the gated segment sum that forms both of its updates (angles -> bonds, edges -> atoms) and
// its VJP, the linear per-atom readout and the geometry VJP that folds every radial gradient.
//
// Gated sum: out[s] (+)= scale * sum_{r in run s} silu(z[r]) * w(r), with the runs of a CSR
// whose rows are the identity (the rows of each segment contiguous: the edges of a centre, the
// triplets of a first bond) and w(r) a per-row weight: w[r], w[i1[r]], or w[i1[r]] w[i2[r]]
// (the two bonds' envelopes of a triplet). One wave per segment, channels across the lanes,
// rows summed in row order: deterministic, no atomics.
#include "common.h"

namespace {

__device__ __forceinline__ float tb_sigmoid(float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

__device__ __forceinline__ int64_t tb_real_rows(const int64_t* n_edges, int64_t e_cap) {
  const int64_t e = n_edges[0];
  return e < e_cap ? e : e_cap;
}

// the polynomial cutoff 1 - 21x^5 + 35x^6 - 15x^7 (x = r / rc) and its r-derivative
__device__ __forceinline__ void poly_cutoff(float r, float rc, float& f, float& df) {
  const float x = r / rc;
  f = 0.f;
  df = 0.f;
  if (x < 1.0f) {
    const float x2 = x * x, x4 = x2 * x2, x5 = x4 * x;
    f = 1.0f - 21.0f * x5 + 35.0f * x5 * x - 15.0f * x5 * x2;
    const float omx = 1.0f - x;
    df = -105.0f * x4 * omx * omx / rc;
  }
}

// geo rows [u_x, u_y, u_z, r, fc, dfc, s, ds]: s = the bond envelope of a short real row
__global__ void tb_envelope_kernel(float* geo, const uint8_t* short_flags, const int64_t* n_edges, int64_t e_cap,
                                   float rb) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= e_cap) return;
  float s = 0.f, ds = 0.f;
  if (e < tb_real_rows(n_edges, e_cap) && short_flags[e]) poly_cutoff(geo[8 * e + 3], rb, s, ds);
  geo[8 * e + 6] = s;
  geo[8 * e + 7] = ds;
}

struct RowWeight {
  const float* w;
  int64_t ldw;
  const int32_t* i1;  // null: w[r]
  const int32_t* i2;  // null: w[i1[r]]
  int64_t ld_idx;
  __device__ __forceinline__ float w1(int64_t r) const { return i1 ? w[(int64_t)i1[r * ld_idx] * ldw] : w[r * ldw]; }
  __device__ __forceinline__ float w2(int64_t r) const { return i2 ? w[(int64_t)i2[r * ld_idx] * ldw] : 1.0f; }
};

__device__ __forceinline__ void run_of(const int64_t* off, int64_t s, int64_t rows, int64_t& lo, int64_t& hi) {
  lo = off[s];
  hi = off[s + 1];
  hi = hi < rows ? hi : rows;
  lo = lo < hi ? lo : hi;
}

// The channel columns of a lane: c = lane + 64 cc (cc < NC); lanes past C read column C - 1 (a
// real column, so every load stays in the row) and store nothing.
template <int NC>
struct LaneCols {
  int col[NC];
  bool live[NC];
  __device__ __forceinline__ explicit LaneCols(int C) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) {
      const int c = lane + 64 * cc;
      live[cc] = c < C;
      col[cc] = c < C ? c : C - 1;
    }
  }
};

// the value of lane j (j wave-uniform)
__device__ __forceinline__ float lane_value(float v, int j) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}

// Rows per batch of the gated sums: a batch's loads (clamped to the run's last row) are all issued
// before its arithmetic, and the rows past the run are masked out of the sums; a run of up to R
// rows costs one memory round trip instead of one per four rows. R = 8 measured faster than 16 at
// one channel per lane (5 000 atoms, 15 edge rows per atom: the partial second batch is cheaper
// than the masked half of a single one, and the waves hold fewer registers).
template <int NC>
constexpr int gated_batch() {
  return 8;
}

template <int NC>
__global__ void __launch_bounds__(256) tb_gated_sum_kernel(const float* z, int64_t ldz, int64_t rows, int C,
                                                            RowWeight rw, const int64_t* off, int64_t n_seg,
                                                            float scale, float* out, int64_t ldo, int accumulate) {
  constexpr int R = gated_batch<NC>();
  const int lane = threadIdx.x & 63;
  const int64_t s = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if (s >= n_seg) return;
  int64_t lo, hi;
  run_of(off, s, rows, lo, hi);
  const LaneCols<NC> lc(C);
  float* o = out + s * ldo;
  float old[NC], acc[NC];
#pragma unroll
  for (int cc = 0; cc < NC; ++cc) {
    old[cc] = accumulate ? o[lc.col[cc]] : 0.f;
    acc[cc] = 0.f;
  }
  for (int64_t r0 = lo; r0 < hi; r0 += R) {
    const int m = hi - r0 >= R ? R : (int)(hi - r0);
    // the batch's row weights one per lane (lane j: row j), read back per row from that lane
    const int64_t rl = r0 + (lane < m ? lane : m - 1);
    const float wl = rw.w1(rl) * rw.w2(rl);
    float x[R][NC];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int64_t r = r0 + (j < m ? j : m - 1);
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) x[j][cc] = z[r * ldz + lc.col[cc]];
    }
    // rows in order; the masked rows leave the sum as it is
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const float w = lane_value(wl, j);
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) {
        const float v = x[j][cc] * tb_sigmoid(x[j][cc]) * w;
        acc[cc] = j < m ? acc[cc] + v : acc[cc];
      }
    }
  }
#pragma unroll
  for (int cc = 0; cc < NC; ++cc)
    if (lc.live[cc]) o[lc.col[cc]] = accumulate ? old[cc] + scale * acc[cc] : scale * acc[cc];
}

// VJP: per row of run s, with g = scale * gout[s]: gz[r] = g w(r) silu'(z[r]) and
// gw(r) = sum_c g silu(z[r]) (the weight's gradient; with two indices written as the two
// envelopes' terms (gw w2, gw w1); added to gw with acc_gw); gsum[s] = sum_r gz[r]. Rows past the
// last run: gz = 0, gw = 0 (left as they are with acc_gw).
template <int NC>
__global__ void __launch_bounds__(256) tb_gated_sum_bwd_kernel(const float* gout, int64_t ldg, const float* z,
                                                                int64_t ldz, int64_t rows, int C, RowWeight rw,
                                                                const int64_t* off, int64_t n_seg, float scale,
                                                                float* gz, int64_t ldgz, float* gsum, int64_t ldgs,
                                                                float* gw, int64_t ldgw, int acc_gw,
                                                                int64_t seg_blocks) {
  constexpr int R = gated_batch<NC>();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if ((int64_t)blockIdx.x >= seg_blocks) {
    // the rows of no segment
    const int64_t tail = off[n_seg] < rows ? off[n_seg] : rows;
    const int64_t step = ((int64_t)gridDim.x - seg_blocks) * 4;
    for (int64_t r = tail + ((int64_t)blockIdx.x - seg_blocks) * 4 + wave; r < rows; r += step) {
      for (int c = lane; c < C; c += 64) gz[r * ldgz + c] = 0.f;
      if (gw && !acc_gw && lane < (rw.i2 ? 2 : 1)) gw[r * ldgw + lane] = 0.f;
    }
    return;
  }
  const int64_t s = (int64_t)blockIdx.x * 4 + wave;
  if (s >= n_seg) return;
  int64_t lo, hi;
  run_of(off, s, rows, lo, hi);
  const LaneCols<NC> lc(C);
  const bool two = rw.i2 != nullptr, old_gw = gw && acc_gw;
  float g[NC], acc[NC];
#pragma unroll
  for (int cc = 0; cc < NC; ++cc) {
    g[cc] = lc.live[cc] ? scale * gout[s * ldg + lc.col[cc]] : 0.f;
    acc[cc] = 0.f;
  }
  for (int64_t r0 = lo; r0 < hi; r0 += R) {
    const int m = hi - r0 >= R ? R : (int)(hi - r0);
    // every load of the batch before its arithmetic: the rows, and one per lane (lane j: row j)
    // the row's weights and old weight gradients, read back per row from that lane
    const int64_t rl = r0 + (lane < m ? lane : m - 1);
    const float wal = rw.w1(rl), wbl = rw.w2(rl);
    const float go0 = old_gw ? gw[rl * ldgw] : 0.f, go1 = old_gw && two ? gw[rl * ldgw + 1] : 0.f;
    float xs[R][NC];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int64_t r = r0 + (j < m ? j : m - 1);
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) xs[j][cc] = z[r * ldz + lc.col[cc]];
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int64_t r = r0 + j;
      const float a = lane_value(wal, j), b = lane_value(wbl, j), w = a * b;
      float p = 0.f, v[NC];
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) {
        const float x = xs[j][cc];
        const float sg = tb_sigmoid(x);
        const float si = x * sg;
        v[cc] = g[cc] * w * (sg + si * (1.0f - sg));
        acc[cc] = j < m ? acc[cc] + v[cc] : acc[cc];
        p += g[cc] * si;  // g = 0 on the lanes past C
      }
      if (j < m) {
#pragma unroll
        for (int cc = 0; cc < NC; ++cc)
          if (lc.live[cc]) gz[r * ldgz + lc.col[cc]] = v[cc];
      }
      if (gw) {
        const float t = wave_sum(p);
        if (j < m && lane == 0) {
          if (two) {
            gw[r * ldgw] = lane_value(go0, j) + t * b;
            gw[r * ldgw + 1] = lane_value(go1, j) + t * a;
          } else {
            gw[r * ldgw] = lane_value(go0, j) + t;
          }
        }
      }
    }
  }
  if (gsum) {
#pragma unroll
    for (int cc = 0; cc < NC; ++cc)
      if (lc.live[cc]) gsum[s * ldgs + lc.col[cc]] = acc[cc];
  }
}

// E_i = e0[elem_i] + h_i . wr
__global__ void __launch_bounds__(256) tb_readout_kernel(const float* h, int64_t ldh, int C, const float* wr,
                                                          const int32_t* elem, const float* e0, int64_t n,
                                                          float* energy) {
  const int lane = threadIdx.x & 63;
  const int64_t i = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if (i >= n) return;
  float p = 0.f;
  for (int c = lane; c < C; c += 64) p += h[i * ldh + c] * wr[c];
  p = wave_sum(p);
  if (lane == 0) energy[i] = e0[elem[i]] + p;
}

// gh_i = g_i wr (g_i = gE[i], or `sign` without gE)
__global__ void tb_readout_bwd_kernel(const float* ge, float sign, const float* wr, int C, int64_t n, float* gh,
                                      int64_t ldgh) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * C) return;
  const int64_t i = t / C;
  const int c = (int)(t - i * C);
  gh[i * ldgh + c] = (ge ? ge[i] : sign) * wr[c];
}

// gvec = gr u + (gu - (gu . u) u) / r with gr = sum_n gef def + gfc dfc + gs ds
struct RowGrads {
  const float *geo, *def, *gef, *gu, *gfc, *gs;
  const uint8_t* bond_flags;
  int64_t ldgef, ldgu;
  int nb;
  bool wide;
  __device__ __forceinline__ void operator()(int64_t e, float (&out)[3]) const {
    const float* g = geo + 8 * e;
    float gr = gef ? basis_dot(def + e * nb, gef + e * ldgef, nullptr, nb, wide) : 0.f;
    if (gfc) gr += gfc[e] * g[5];
    // gs and gu hold values on the bond rows only (with bond_flags; else on every row)
    const bool bond = bond_flags ? bond_flags[e] != 0 : true;
    if (gs && bond) gr += gs[e] * g[7];
    float v[3] = {0.f, 0.f, 0.f};
    if (gu && bond) {
      v[0] = gu[e * ldgu];
      v[1] = gu[e * ldgu + 1];
      v[2] = gu[e * ldgu + 2];
    }
    const float inv_r = 1.0f / g[3];
    const float gdotu = v[0] * g[0] + v[1] * g[1] + v[2] * g[2];
#pragma unroll
    for (int k = 0; k < 3; ++k) out[k] = gr * g[k] + (v[k] - gdotu * g[k]) * inv_r;
  }
};

__global__ void tb_geometry_bwd_kernel(const RowGrads rg, const int64_t* n_edges, int64_t e_cap, float* gvec) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= e_cap) return;
  if (e >= tb_real_rows(n_edges, e_cap)) {
    gvec[3 * e] = gvec[3 * e + 1] = gvec[3 * e + 2] = 0.f;
    return;
  }
  float v[3];
  rg(e, v);
#pragma unroll
  for (int k = 0; k < 3; ++k) gvec[3 * e + k] = v[k];
}

// the forces straight from them (edge_forces_of): 8.3 + 6.0 us of the row kernel and the segment sum -> 6.8 at
// 5 000 atoms
__global__ void __launch_bounds__(256) tb_edge_forces_kernel(const RowGrads rg, const int64_t* off,
                                                             const int32_t* reverse, const int64_t* n_edges,
                                                             int64_t e_cap, int64_t n, float sign, float* forces,
                                                             float* gvec) {
  const int64_t i = fmd_xcd_block(blockIdx.x, gridDim.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if (i < n) edge_forces_of(i, off, reverse, tb_real_rows(n_edges, e_cap), sign, forces, gvec, rg);
}

// ---- angle -> bond sums over the line graph. The work is a few bonds and triplets per atom, far
// fewer than the edge rows: each kernel runs a fixed grid of waves that strides over the real
// bonds (bond_rows[0, short_offsets[n])) or triplets ([0, pair_offsets[n])), counts read on the
// device, several bonds or triplets per wave and pass (channels across the lanes) whose loads are
// all issued before their arithmetic: one chain of dependent loads per pass, not per item. A
// bond's triplets as first bond are the run [eto[b], eto[b+1]) of the line graph (contiguous), as
// second bond the same run through second_perm.
struct LineCsr {
  const int64_t* short_offsets;  // [n + 1]: the bond count at [n]
  const int32_t* bond_rows;      // [e_cap]
  const int64_t* eto;            // edge_triplet_offsets [e_cap + 1]
  const int32_t* second_perm;    // [t_cap]
  const int32_t* line;           // line_graph [t_cap, 5]: (atom, pair 1, row 1, pair 2, row 2)
  const int64_t* pair_offsets;   // [n + 1]: the triplet count at [n]
  int64_t n;
  int64_t t_cap;
};

constexpr int kStrideBlocks = 1024;  // 4096 waves (about four per SIMD)

__device__ __forceinline__ int64_t wave_id() {
  return (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
}

// The index work of a pass runs across the lanes (one load instruction per level of the chain
// bond_rows -> eto -> line graph / second_perm -> envelope for all of the pass's bonds or
// triplets), the channel rows across the wave with the indices read back per lane: a pass costs
// one chain of dependent loads, whatever the number of bonds or triplets in it.
__device__ __forceinline__ int lane_int(int v, int j) { return __builtin_amdgcn_readlane(v, j); }

// Lane q < U: bond slot q of the pass (bond j0 + q NW of bond_rows; past the count the pass's
// first bond again, loaded and not stored) with its run [lo, hi) of triplets as first bond,
// clamped to t_cap.
template <int U>
struct BondSlots {
  int b, lo, hi;
  bool ok;
  __device__ __forceinline__ BondSlots(const LineCsr& lc, int64_t j0, int64_t nw, int64_t nb) {
    const int lane = threadIdx.x & 63;
    const int64_t j = j0 + (lane < U ? lane : 0) * nw;
    ok = j < nb;
    b = lc.bond_rows[ok ? j : j0];
    int64_t l = lc.eto[b], h = lc.eto[(int64_t)b + 1];
    h = h < lc.t_cap ? h : lc.t_cap;
    l = l < h ? l : h;
    lo = (int)l;
    hi = (int)h;
  }
  __device__ __forceinline__ int64_t bond(int q) const { return lane_int(b, q); }
  __device__ __forceinline__ int64_t count(int q) const { return lane_int(hi, q) - lane_int(lo, q); }
  __device__ __forceinline__ bool stored(int q) const { return lane_int(ok ? 1 : 0, q) != 0; }
  // on lane l: triplet t of bond q's run, clamped to its last triplet (row 0 for an empty run,
  // whose loads are then not used as addresses)
  __device__ __forceinline__ int64_t slot_row(int q, int t, bool& empty) const {
    const int l = __shfl(lo, q, 64), h = __shfl(hi, q, 64);
    empty = h <= l;
    return l + t < h ? l + t : (h > l ? h - 1 : 0);
  }
};

// bonds per pass and triplets per bond whose loads go out together (longer runs finish in a loop)
template <int NC>
constexpr int bond_pass() {
  return NC == 1 ? 4 : 2;
}
constexpr int kRunBatch = 4;

// The pre-activation of a triplet from its bonds' and its atom's rows: z3[k] = u[b1] + v[b2] + h[atom] + aw[k].
struct TripletTerms {
  const float* u;  // [e_cap] rows (bond rows only), row stride ldu
  const float* v;
  const float* h;   // [n] rows, row stride ldh
  const float* aw;  // [t_cap] rows, row stride lda
  int64_t ldu, ldh, lda;
};

// eps[b] += scale * sum over b's triplets (first bond), in order, of silu(z3[k]) s_b s_b2; z3 is formed here
// from its four rows and stored for the VJP.
template <int NC>
__global__ void __launch_bounds__(256) tb_bond_sum_kernel(LineCsr lc, float* z3, int64_t ldz, int C,
                                                           const TripletTerms tt, const float* geo, float scale,
                                                           float* eps, int64_t lde) {
  constexpr int U = bond_pass<NC>(), TQ = kRunBatch;
  const int lane = threadIdx.x & 63;
  const LaneCols<NC> cols(C);
  const int64_t nb = lc.short_offsets[lc.n], nw = (int64_t)gridDim.x * 4;
  for (int64_t j0 = wave_id(); j0 < nb; j0 += U * nw) {
    const BondSlots<U> bs(lc, j0, nw, nb);
    float old[U][NC], x[U][TQ][NC];
#pragma unroll
    for (int q = 0; q < U; ++q)
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) old[q][cc] = eps[bs.bond(q) * lde + cols.col[cc]];
    // lane l < U TQ: triplet slot (l / TQ, l % TQ) and its weight s_b s_b2
    const int qs = lane < U * TQ ? lane / TQ : 0;
    bool empty;
    const int64_t ks = bs.slot_row(qs, lane % TQ, empty);
    const int b2raw = lc.line[5 * ks + 4];
    const int bq = __shfl(bs.b, qs, 64);
    const int b2 = empty ? bq : b2raw;  // an empty run's slots read the bond's own rows and add nothing
    float ub[U][NC];
    const int atom_l = empty ? 0 : lc.line[5 * ks];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int64_t at = lane_int(atom_l, q * TQ);
#pragma unroll
      for (int cc = 0; cc < NC; ++cc)
        ub[q][cc] = tt.u[bs.bond(q) * tt.ldu + cols.col[cc]] + tt.h[at * tt.ldh + cols.col[cc]];
    }
#pragma unroll
    for (int q = 0; q < U; ++q)
#pragma unroll
      for (int t = 0; t < TQ; ++t) {
        const int64_t k = lane_int((int)ks, q * TQ + t);
        const int64_t r2 = lane_int(b2, q * TQ + t);
#pragma unroll
        for (int cc = 0; cc < NC; ++cc)
          x[q][t][cc] = tt.aw[k * tt.lda + cols.col[cc]] + tt.v[r2 * tt.ldu + cols.col[cc]];
      }
    const float w1 = geo[8 * (int64_t)bq + 6];
    const float ws = w1 * geo[8 * (int64_t)b2 + 6];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      float acc[NC];
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) acc[cc] = 0.f;
      const int64_t cnt = bs.count(q);
#pragma unroll
      for (int t = 0; t < TQ; ++t) {
        const float w = lane_value(ws, q * TQ + t);
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) {
          const float z = x[q][t][cc] + ub[q][cc];
          if (t < cnt && bs.stored(q) && cols.live[cc])
            z3[(int64_t)lane_int((int)ks, q * TQ + t) * ldz + cols.col[cc]] = z;
          const float v = z * tb_sigmoid(z) * w;
          acc[cc] = t < cnt ? acc[cc] + v : acc[cc];
        }
      }
      // the rest of a longer run, four triplets' loads at a time
      const int64_t lo = lane_int(bs.lo, q), hi = lane_int(bs.hi, q);
      const float w1q = lane_value(w1, q * TQ);
      for (int64_t k0 = lo + TQ; k0 < hi; k0 += 4) {
        const int m = hi - k0 >= 4 ? 4 : (int)(hi - k0);
        float y[4][NC], wy[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int64_t k = k0 + (t < m ? t : m - 1);
          const int64_t r2 = lc.line[5 * k + 4];
          wy[t] = w1q * geo[8 * r2 + 6];
#pragma unroll
          for (int cc = 0; cc < NC; ++cc)
            y[t][cc] = tt.aw[k * tt.lda + cols.col[cc]] + tt.v[r2 * tt.ldu + cols.col[cc]];
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int cc = 0; cc < NC; ++cc) {
            const float z = y[t][cc] + ub[q][cc];
            if (t < m && bs.stored(q) && cols.live[cc]) z3[(k0 + t) * ldz + cols.col[cc]] = z;
            const float v = z * tb_sigmoid(z) * wy[t];
            acc[cc] = t < m ? acc[cc] + v : acc[cc];
          }
      }
      if (bs.stored(q)) {
        const int64_t b = bs.bond(q);
#pragma unroll
        for (int cc = 0; cc < NC; ++cc)
          if (cols.live[cc]) eps[b * lde + cols.col[cc]] = old[q][cc] + scale * acc[cc];
      }
    }
  }
}

// triplets per pass of the triplet VJP
template <int NC>
constexpr int triplet_pass() {
  return NC == 1 ? 8 : 4;
}

// Per triplet k: with g = scale geps[b1], gz3[k] = g s_b1 s_b2 silu'(z3[k]) and
// gw = sum_c g silu(z3[k]), stored as the envelope terms gsw[k] = (gw s_b2, gw s_b1). Rows past
// the real triplets: gz3 = 0.
template <int NC>
__global__ void __launch_bounds__(256) tb_triplet_bwd_kernel(LineCsr lc, const float* geps, int64_t ldg,
                                                              const float* z3, int64_t ldz, int C, const float* geo,
                                                              float scale, float* gz3, int64_t ldgz, float* gsw) {
  constexpr int U = triplet_pass<NC>();
  const int lane = threadIdx.x & 63;
  const LaneCols<NC> cols(C);
  const int64_t t_all = lc.pair_offsets[lc.n];
  const int64_t t_real = t_all < lc.t_cap ? t_all : lc.t_cap;
  const int64_t nw = (int64_t)gridDim.x * 4;
  for (int64_t k0 = wave_id(); k0 < lc.t_cap; k0 += U * nw) {
    // lane q < U: triplet slot q (k0 + q NW); a slot past the real triplets loads line-graph row 0
    // and edge row 0 (in bounds, unused)
    const int64_t kl = k0 + (lane < U ? lane : 0) * nw;
    const bool real = kl < t_real;
    const int64_t kr = real ? kl : 0;
    const int r1 = lc.line[5 * kr + 2], r2 = lc.line[5 * kr + 4];
    float x[U][NC], g[U][NC];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int64_t kq = k0 + q * nw < t_real ? k0 + q * nw : 0;
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) x[q][cc] = z3[kq * ldz + cols.col[cc]];
    }
    const int b1 = real ? r1 : 0, b2 = real ? r2 : 0;
    const float w1l = geo[8 * (int64_t)b1 + 6], w2l = geo[8 * (int64_t)b2 + 6];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int64_t b = lane_int(b1, q);
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) g[q][cc] = scale * geps[b * ldg + cols.col[cc]];
    }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int64_t kq = k0 + q * nw;
      if (kq >= lc.t_cap) continue;
      float* out = gz3 + kq * ldgz;
      if (kq >= t_real) {
#pragma unroll
        for (int cc = 0; cc < NC; ++cc)
          if (cols.live[cc]) out[cols.col[cc]] = 0.f;
        continue;
      }
      const float w1 = lane_value(w1l, q), w2 = lane_value(w2l, q), w = w1 * w2;
      float p = 0.f;
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) {
        const float sg = tb_sigmoid(x[q][cc]);
        const float si = x[q][cc] * sg;
        if (cols.live[cc]) {
          out[cols.col[cc]] = g[q][cc] * w * (sg + si * (1.0f - sg));
          p += g[q][cc] * si;
        }
      }
      const float gw = wave_sum(p);
      if (lane == 0) {
        gsw[2 * kq] = gw * w2;
        gsw[2 * kq + 1] = gw * w1;
      }
    }
  }
}

// Per bond b: guv[b, 0:C] = sum of gz3 [t_cap, C] (the gradient of z3) over b's triplets as first bond, guv[b, C:2C] as
// second bond; gs[b] (+)= the same sums of gsw[k, 0] and gsw[k, 1] (stored, or added with acc_gs). A
// second-bond slot of -1 (no triplet) adds zeros.
template <int NC>
__device__ __forceinline__ void bond_sums(const LineCsr& lc, const float* gz3, int64_t ldz, int C, const float* gsw,
                                          float* guv, int64_t ldg, float* gs, int acc_gs, int64_t first_wave,
                                          int64_t nw) {
  constexpr int U = bond_pass<NC>(), TQ = kRunBatch;
  const int lane = threadIdx.x & 63;
  const LaneCols<NC> cols(C);
  const int64_t nb = lc.short_offsets[lc.n];
  for (int64_t j0 = first_wave; j0 < nb; j0 += U * nw) {
    const BondSlots<U> bs(lc, j0, nw, nb);
    const float gs_l = acc_gs ? gs[bs.b] : 0.f;
    float x[U][2][TQ][NC];
    // lane l < 2 U TQ: role l / (U TQ), slot ((l % U TQ) / TQ, l % TQ); role 1 through second_perm
    const int sl = lane % (U * TQ), role_l = lane < U * TQ ? 0 : 1;
    bool empty;
    const int64_t pl = bs.slot_row(lane < 2 * U * TQ ? sl / TQ : 0, sl % TQ, empty);
    const int sp = lc.second_perm[pl];
#pragma unroll
    for (int q = 0; q < U; ++q)
#pragma unroll
      for (int t = 0; t < TQ; ++t) {
        const int64_t k = lane_int((int)pl, q * TQ + t);
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) x[q][0][t][cc] = gz3[k * ldz + cols.col[cc]];
      }
    const int kk = role_l == 0 ? (int)pl : (empty ? -1 : sp);
    const float sw = gsw[2 * (int64_t)(kk >= 0 ? kk : 0) + role_l];
#pragma unroll
    for (int q = 0; q < U; ++q)
#pragma unroll
      for (int t = 0; t < TQ; ++t) {
        const int k = lane_int(kk, U * TQ + q * TQ + t);
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) x[q][1][t][cc] = gz3[(int64_t)(k >= 0 ? k : 0) * ldz + cols.col[cc]];
      }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      float acc[NC], gsum = 0.f;
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) acc[cc] = 0.f;
      const int64_t cnt = bs.count(q), lo = lane_int(bs.lo, q), hi = lane_int(bs.hi, q);
#pragma unroll
      for (int role = 0; role < 2; ++role) {
#pragma unroll
        for (int t = 0; t < TQ; ++t) {
          const int l = role * U * TQ + q * TQ + t;
          const bool use = t < cnt, ok = lane_int(kk, l) >= 0;
#pragma unroll
          for (int cc = 0; cc < NC; ++cc) {
            const float v = ok ? x[q][role][t][cc] : 0.f;
            acc[cc] = use ? acc[cc] + v : acc[cc];
          }
          const float v = ok ? lane_value(sw, l) : 0.f;
          gsum = use ? gsum + v : gsum;
        }
        // the rest of a longer run, four slots' loads at a time
        for (int64_t p0 = lo + TQ; p0 < hi; p0 += 4) {
          const int m = hi - p0 >= 4 ? 4 : (int)(hi - p0);
          int64_t ky[4];
          float y[4][NC], sy[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int64_t p = p0 + (t < m ? t : m - 1);
            ky[t] = role == 0 ? p : (int64_t)lc.second_perm[p];
          }
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int64_t k = ky[t] >= 0 ? ky[t] : 0;
            sy[t] = gsw[2 * k + role];
#pragma unroll
            for (int cc = 0; cc < NC; ++cc) y[t][cc] = gz3[k * ldz + cols.col[cc]];
          }
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const bool use = t < m, ok = ky[t] >= 0;
#pragma unroll
            for (int cc = 0; cc < NC; ++cc) {
              const float v = ok ? y[t][cc] : 0.f;
              acc[cc] = use ? acc[cc] + v : acc[cc];
            }
            const float v = ok ? sy[t] : 0.f;
            gsum = use ? gsum + v : gsum;
          }
        }
        if (bs.stored(q)) {
          float* out = guv + bs.bond(q) * ldg + role * C;
#pragma unroll
          for (int cc = 0; cc < NC; ++cc)
            if (cols.live[cc]) out[cols.col[cc]] = acc[cc];
        }
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) acc[cc] = 0.f;
      }
      if (bs.stored(q) && lane == 0) gs[bs.bond(q)] = lane_value(gs_l, q) + gsum;
    }
  }
}

// out[c] = sum over entries [lo, hi) of row perm[k] (null: row k; negative: none) of v, a wave: G groups of C / 4
// lanes take the entries in turn, U of each group's rows in flight, the groups added in a fixed order.
template <int NC>
__device__ __forceinline__ void row_sums(const float* v, int64_t ld, const int32_t* perm, int64_t lo, int64_t hi,
                                         float* out) {
  constexpr int LPR = 16 * NC, G = NC == 1 ? 4 : NC == 2 ? 2 : 1, U = NC == 1 ? 5 : 8;
  const int lane = threadIdx.x & 63, g = G == 1 ? 0 : lane / LPR, c = 4 * (lane - g * LPR);
  const bool live = lane < G * LPR;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int64_t base = lo; base < hi; base += 64) {
    const int cnt = hi - base < 64 ? (int)(hi - base) : 64;
    const int64_t k = base + (lane < cnt ? lane : cnt - 1);
    const int row = perm ? perm[k] : (int)k;
    for (int k0 = 0; k0 < cnt; k0 += G * U) {
      float4 x[U];
      bool use[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int at = k0 + u * G + g, r = __shfl(row, at < cnt ? at : cnt - 1, 64);
        use[u] = at < cnt && r >= 0;
        x[u] = *reinterpret_cast<const float4*>(v + (int64_t)(r >= 0 ? r : 0) * ld + (live ? c : 0));
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        acc.x = use[u] ? acc.x + x[u].x : acc.x;
        acc.y = use[u] ? acc.y + x[u].y : acc.y;
        acc.z = use[u] ? acc.z + x[u].z : acc.z;
        acc.w = use[u] ? acc.w + x[u].w : acc.w;
      }
    }
  }
#pragma unroll
  for (int s = LPR; s < LPR * G; s *= 2) {
    acc.x += __shfl_xor(acc.x, s, 64);
    acc.y += __shfl_xor(acc.y, s, 64);
    acc.z += __shfl_xor(acc.z, s, 64);
    acc.w += __shfl_xor(acc.w, s, 64);
  }
  if (live && g == 0) *reinterpret_cast<float4*>(out + c) = acc;
}

struct NodeSums {
  const float* gz2;        // [e_cap, C]
  const int64_t* off;      // [n + 1]
  const int32_t* reverse;  // [e_cap]: the rows sent by an atom
  int64_t e_cap;
  float *src, *tri;        // [n] rows of stride ld
  int64_t ld;
};

// The sums that a layer's VJP forms once gz2 and gz3 are there, none of which reads another: per bond [gU | gV] and
// the envelope terms (the first blocks: the longest chain), per atom the gz2 of the edges that it sends and the gz3
// of its triplets. One launch instead of three:
// 13.8 us against 12.5 + 8 + 4.7 at 5 000 atoms and 64 channels (MD step 698 -> 647 us; 375 atoms, 128 channels 470 ->
// 422).
template <int NC>
__global__ void __launch_bounds__(256) tb_vjp_sums_kernel(LineCsr lc, const float* gz3, int64_t ldz, int C,
                                                           const float* gsw, float* guv, int64_t ldg, float* gs,
                                                           int acc_gs, const NodeSums ns, int64_t bond_blocks) {
  if ((int64_t)blockIdx.x < bond_blocks) {
    bond_sums<NC>(lc, gz3, ldz, C, gsw, guv, ldg, gs, acc_gs, wave_id(), bond_blocks * 4);
    return;
  }
  const int64_t w = wave_id() - bond_blocks * 4, i = w >> 1;
  if (i >= lc.n) return;
  int64_t lo, hi;
  if (w & 1) {
    run_of(lc.pair_offsets, i, lc.t_cap, lo, hi);
    row_sums<NC>(gz3, ldz, nullptr, lo, hi, ns.tri + i * ns.ld);
  } else {
    run_of(ns.off, i, ns.e_cap, lo, hi);
    row_sums<NC>(ns.gz2, C, ns.reverse, lo, hi, ns.src + i * ns.ld);
  }
}

// ---- the bond rows' products and the edge sums of the node-factored model. An edge row's pre-activation
// z2 = h_j W2a + h_i W2b + eps_e W2c takes its first two terms from per-atom rows, and eps_e differs from
// its initial ef_e We on the bond rows alone (a tenth of the edges): the other rows' last term is
// ef_e (We W2c), an nb-term sum formed here per row, and the products with C x C blocks run on the
// bond rows only. No edge-sized product and no triplet-sized one is left (5 000 atoms, 3.5 A: 84 000
// edges, 10 300 bonds, 26 000 triplets).
// Against gathering [h_j | eps_e] and [eps_b1 | eps_b2 | h_i] into products over the edge and triplet rows: an MD step
// of 5 000 atoms at 64 channels 773 -> 698 us, of 375 atoms at 128 channels 767 -> 470, an evaluation of 500
// atoms 988 -> 574 (then 647, 422 and 550 with the sums above in one launch).

// C[e, 0:N] (+)= [a0[e] | a1[e]] B^T over the real bonds e = bond_rows[k]: a workgroup takes 16 bonds x 64 columns,
// each wave one 16 x 16 block of v_mfma_f32_16x16x4_f32 with its operands straight into registers (lane group
// g = l / 16 holds k = 8 g .. 8 g + 8 of a 32-k slice), the loads of up to four slices in flight: the operands are
// one round trip per 128 of K behind the row look-up. The count is read on the device, the grid strides. Bound by that
// chain of round trips: 7.9 us at 400 atoms and 128 channels (12.4 with one wave per 16 x 64 tile and one
// slice in flight), 11.4 at 10 300 bonds and 64 channels (the same). S: the slices in flight, two where K has no
// more (fewer registers, seven waves per SIMD instead of four: K = 64 at 10 300 bonds 11.4 -> 10.5 us).
typedef float f32x4_t __attribute__((ext_vector_type(4)));

struct BondProduct {
  const float *a0, *a1, *b;
  float* c;
  int64_t ld0, ld1, ldb, ldc;
  int k0, k, n, accumulate;  // columns [0, k0) of K from a0, the rest from a1
  const uint8_t* overflow;   // nullable: the build's flag
};

// An overflowed build's bond rows and triplet rows do not belong together (its triplets are the padding topology's),
// and rows that no kernel below writes may be read: what would be their products is zero on every row instead, so
// that such an evaluation, whose results are discarded, is finite whatever the memory held.
__device__ __forceinline__ void zero_rows(float* c, int64_t ldc, int64_t rows, int n) {
  const int64_t step = (int64_t)gridDim.x * 4;
  for (int64_t r = wave_id(); r < rows; r += step)
    for (int k = threadIdx.x & 63; k < n; k += 64) c[r * ldc + k] = 0.f;
}

__device__ __forceinline__ int64_t bond_count(const LineCsr& lc, int64_t e_cap) {
  const int64_t nb = lc.short_offsets[lc.n];
  return nb < e_cap ? nb : e_cap;
}

template <int S>
__global__ void __launch_bounds__(256) tb_bond_product_kernel(LineCsr lc, int64_t e_cap, const BondProduct p) {
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int64_t nb = bond_count(lc, e_cap), nw = (int64_t)gridDim.x * 4;
  if (p.overflow && p.overflow[0]) {
    if (!p.accumulate) zero_rows(p.c, p.ldc, e_cap, p.n);
    return;
  }
  const int64_t ct = p.n / 16, tiles = fmd_cdiv(nb, 16) * ct;  // a multiple of four: a workgroup's waves share bonds
  for (int64_t w = wave_id(); w < tiles; w += nw) {
    const int64_t tm = w / ct, col = (w - tm * ct) * 16 + i, slot = tm * 16 + i;
    const int e = lc.bond_rows[slot < nb ? slot : nb - 1];
    const float *r0 = p.a0 + e * p.ld0, *r1 = p.a1 ? p.a1 + e * p.ld1 : r0, *bp = p.b + col * p.ldb + 8 * g;
    f32x4_t acc{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < p.k; k0 += 32 * S) {
      float4 a[S][2], b[S][2];
#pragma unroll
      for (int q = 0; q < S; ++q) {
        const int k = k0 + 32 * q;
        if (k >= p.k) break;
        b[q][0] = *reinterpret_cast<const float4*>(bp + k);
        b[q][1] = *reinterpret_cast<const float4*>(bp + k + 4);
        const float* ap = (k < p.k0 ? r0 + k : r1 + (k - p.k0)) + 8 * g;
        a[q][0] = *reinterpret_cast<const float4*>(ap);
        a[q][1] = *reinterpret_cast<const float4*>(ap + 4);
      }
#pragma unroll
      for (int q = 0; q < S; ++q) {
        if (k0 + 32 * q >= p.k) break;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q][h].x, b[q][h].x, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q][h].y, b[q][h].y, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q][h].z, b[q][h].z, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q][h].w, b[q][h].w, acc, 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t row = __shfl(e, 4 * g + v, 64);
      if (tm * 16 + 4 * g + v >= nb) continue;
      float* c = p.c + row * p.ldc + col;
      *c = p.accumulate ? *c + acc[v] : acc[v];
    }
  }
}

// The bond rows' first values: out[e, block b] = ef[e] m[:, b C : (b + 1) C] for the three blocks of m [nb, 3 C],
// stored at columns 0, 2 C and 3 C of the row (eps | . | u | v). A wave takes four bonds and 64 columns, eight rows
// of m in flight together with the bond rows they do not depend on.
__global__ void __launch_bounds__(256) tb_bond_init_kernel(LineCsr lc, int64_t e_cap, const float* ef, int nbasis,
                                                           const float* m, int C, const uint8_t* overflow, float* out,
                                                           int64_t ldo) {
  if (overflow && overflow[0]) {
    zero_rows(out, ldo, e_cap, 4 * C);
    return;
  }
  const int lane = threadIdx.x & 63, blocks = fmd_cdiv(3 * C, 64);
  const int64_t nb = bond_count(lc, e_cap), nw = (int64_t)gridDim.x * 4;
  for (int64_t w = wave_id(); w < fmd_cdiv(nb, 4) * blocks; w += nw) {
    const int64_t j0 = w / blocks * 4;
    const int c = (int)(w % blocks) * 64 + lane, col = c < 3 * C ? c : 3 * C - 1;
    // lane l: bond l / 16, its basis values n0 + l % 16
    const int64_t j = j0 + (lane >> 4);
    const int mine = lc.bond_rows[j < nb ? j : nb - 1];
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int n0 = 0; n0 < nbasis; n0 += 8) {
      float wm[8];
#pragma unroll
      for (int n = 0; n < 8; ++n) wm[n] = n0 + n < nbasis ? m[(int64_t)(n0 + n) * 3 * C + col] : 0.f;
      const int nl = n0 + (lane & 7);
      const float f = nl < nbasis ? ef[(int64_t)mine * nbasis + nl] : 0.f;
#pragma unroll
      for (int n = 0; n < 8; ++n)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] += lane_value(f, 16 * q + n) * wm[n];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (j0 + q < nb && c < 3 * C) out[(int64_t)lane_int(mine, 16 * q) * ldo + (c < C ? c : c + C)] = acc[q];
  }
}

// gef[e, n] = sum_c geps[e, c] We[n, c] on the bond rows (over what the edge kernel left there).
template <int NC>
__global__ void __launch_bounds__(256) tb_bond_basis_kernel(LineCsr lc, int64_t e_cap, const float* geps, int64_t ldg,
                                                            int C, const float* we, int nbasis, float* gef) {
  const int lane = threadIdx.x & 63, idx = wave_sum8_index(lane);
  const LaneCols<NC> lcol(C);
  const int64_t nb = bond_count(lc, e_cap), nw = (int64_t)gridDim.x * 4;
  for (int64_t j = wave_id(); j < nb; j += nw) {
    const int64_t e = lc.bond_rows[j];
    float g[NC];
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) g[cc] = lcol.live[cc] ? geps[e * ldg + lcol.col[cc]] : 0.f;
    for (int n0 = 0; n0 < nbasis; n0 += 8) {
      float v[8];
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        v[n] = 0.f;
#pragma unroll
        for (int cc = 0; cc < NC; ++cc)
          v[n] += n0 + n < nbasis ? g[cc] * we[(int64_t)(n0 + n) * C + lcol.col[cc]] : 0.f;
      }
      const float t = wave_sum8(v);
      if ((lane & 7) == 0 && n0 + idx < nbasis) gef[e * nbasis + n0 + idx] = t;
    }
  }
}

// The edge rows of the sums below.
struct EdgeRows {
  const int64_t* off;  // [n + 1]: the rows of each centre
  int64_t rows, n;
  int C, nb;
  const float* geo;  // column 4: the cutoff, the row's weight
  const float* ef;   // [rows, nb]
  const float* rt;   // [nb, C] = We W2c
};

// 8 basis values of 8 rows across the lanes: lane l holds value n0 + l % 8 of row r0 + l / 8 (clamped to m rows)
__device__ __forceinline__ float basis_lanes(const EdgeRows& er, int64_t r0, int m, int n0) {
  const int lane = threadIdx.x & 63, n = n0 + (lane & 7);
  const int64_t r = r0 + ((lane >> 3) < m ? (lane >> 3) : m - 1);
  return n < er.nb ? er.ef[r * er.nb + n] : 0.f;
}

template <int NC>
__device__ __forceinline__ void basis_weights(const EdgeRows& er, int n0, const LaneCols<NC>& lc, float (&w)[8][NC]) {
#pragma unroll
  for (int n = 0; n < 8; ++n)
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) w[n][cc] = n0 + n < er.nb ? er.rt[(int64_t)(n0 + n) * er.C + lc.col[cc]] : 0.f;
}

// h[i] += scale * sum over i's rows of silu(z2) fc, z2 = p[j] + q[i] + (bond row: xb[e], else ef_e rt), stored for
// the VJP. One wave per centre, batches of 8 rows with their loads issued together (as the gated sums). ONE: nb
// <= 8, the basis weights stay in registers. Bound by the gathered rows' round trips and the z2 stream (21 MB at
// 84 000 rows).
template <int NC, bool ONE>
__global__ void __launch_bounds__(256) tb_edge_sum_kernel(const EdgeRows er, const float* pq, int64_t ldp,
                                                          const int32_t* ei, const uint8_t* flags, const float* xb,
                                                          int64_t ldx, float scale, float* z2, float* h, int64_t ldh) {
  constexpr int R = 8;
  const int lane = threadIdx.x & 63;
  const int64_t s = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if (s >= er.n) return;
  int64_t lo, hi;
  run_of(er.off, s, er.rows, lo, hi);
  const LaneCols<NC> lc(er.C);
  float old[NC], acc[NC], q[NC], w[8][NC];
#pragma unroll
  for (int cc = 0; cc < NC; ++cc) {
    old[cc] = h[s * ldh + lc.col[cc]];
    q[cc] = pq[s * ldp + er.C + lc.col[cc]];
    acc[cc] = 0.f;
  }
  if constexpr (ONE) basis_weights<NC>(er, 0, lc, w);
  for (int64_t r0 = lo; r0 < hi; r0 += R) {
    const int m = hi - r0 >= R ? R : (int)(hi - r0);
    const int64_t rl = r0 + (lane < m ? lane : m - 1);
    const int nbr = ei[2 * rl + 1];
    const float fc = er.geo[8 * rl + 4];
    const int bond = flags[rl];
    float efl = basis_lanes(er, r0, m, 0);
    float z[R][NC], xr[R][NC];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const float* pr = pq + (int64_t)lane_int(nbr, j) * ldp;
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) z[j][cc] = pr[lc.col[cc]];
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) xr[j][cc] = 0.f;
      if (lane_int(bond, j)) {
        const float* x = xb + (r0 + (j < m ? j : m - 1)) * ldx;
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) xr[j][cc] = x[lc.col[cc]];
      }
    }
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) z[j][cc] = (z[j][cc] + q[cc]) + xr[j][cc];
    for (int n0 = 0; n0 < er.nb; n0 += 8) {
      if constexpr (!ONE) {
        basis_weights<NC>(er, n0, lc, w);
        if (n0 > 0) efl = basis_lanes(er, r0, m, n0);
      }
#pragma unroll
      for (int j = 0; j < R; ++j) {
        if (lane_int(bond, j)) continue;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          const float f = lane_value(efl, 8 * j + n);
#pragma unroll
          for (int cc = 0; cc < NC; ++cc) z[j][cc] += f * w[n][cc];
        }
      }
      if constexpr (ONE) break;
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const float f = lane_value(fc, j);
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) {
        if (j < m && lc.live[cc]) z2[(r0 + j) * er.C + lc.col[cc]] = z[j][cc];
        const float v = z[j][cc] * tb_sigmoid(z[j][cc]) * f;
        acc[cc] = j < m ? acc[cc] + v : acc[cc];
      }
    }
  }
#pragma unroll
  for (int cc = 0; cc < NC; ++cc)
    if (lc.live[cc]) h[s * ldh + lc.col[cc]] = old[cc] + scale * acc[cc];
}

// Its VJP: with g = scale gh[i] per row gz2 = g fc silu'(z2), gfc (+)= sum_c g silu(z2), gef[r, n] (+)= sum_c gz2 rt[n]
// (the basis gradient of the rows that are no bonds; the bond rows' is overwritten at the end), per centre
// gsum = sum of gz2. The rows' sums are kept on their lanes and stored once per batch.
template <int NC, bool ONE>
__global__ void __launch_bounds__(256) tb_edge_sum_bwd_kernel(const EdgeRows er, const float* gh, int64_t ldg,
                                                              const float* z2, float scale, float* gz, float* gsum,
                                                              int64_t ldgs, float* gfc, float* gef, int add) {
  constexpr int R = 8;
  const int lane = threadIdx.x & 63, idx = wave_sum8_index(lane), row = lane & 7;
  const int64_t s = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if (s >= er.n) return;
  int64_t lo, hi;
  run_of(er.off, s, er.rows, lo, hi);
  const LaneCols<NC> lc(er.C);
  float g[NC], acc[NC], w[8][NC];
#pragma unroll
  for (int cc = 0; cc < NC; ++cc) {
    g[cc] = lc.live[cc] ? scale * gh[s * ldg + lc.col[cc]] : 0.f;
    acc[cc] = 0.f;
  }
  if constexpr (ONE) basis_weights<NC>(er, 0, lc, w);
  for (int64_t r0 = lo; r0 < hi; r0 += R) {
    const int m = hi - r0 >= R ? R : (int)(hi - r0);
    const int64_t rl = r0 + (lane < m ? lane : m - 1);
    const float fc = er.geo[8 * rl + 4];
    const float old_fc = add ? gfc[rl] : 0.f;
    const bool mine = row < m;
    float v[R][NC];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int64_t r = r0 + (j < m ? j : m - 1);
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) v[j][cc] = z2[r * er.C + lc.col[cc]];
    }
    float sums = 0.f;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const float f = lane_value(fc, j);
      float p = 0.f;
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) {
        const float x = v[j][cc], sg = tb_sigmoid(x), si = x * sg;
        p += g[cc] * si;
        v[j][cc] = g[cc] * f * (sg + si * (1.0f - sg));
        acc[cc] = j < m ? acc[cc] + v[j][cc] : acc[cc];
        if (j < m && lc.live[cc]) gz[(r0 + j) * er.C + lc.col[cc]] = v[j][cc];
      }
      const float t = wave_sum(p);
      sums = lane == j ? t : sums;
    }
    if (lane < m) gfc[rl] = old_fc + sums;
    for (int n0 = 0; n0 < er.nb; n0 += 8) {
      if constexpr (!ONE) basis_weights<NC>(er, n0, lc, w);
      const bool use = mine && n0 + idx < er.nb;
      float* ge = gef + (r0 + (mine ? row : m - 1)) * er.nb + (n0 + idx < er.nb ? n0 + idx : 0);
      const float old = add && use ? *ge : 0.f;
      float got = 0.f;
#pragma unroll
      for (int j = 0; j < R; ++j) {
        float d[8];
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          d[n] = 0.f;
#pragma unroll
          for (int cc = 0; cc < NC; ++cc) d[n] += v[j][cc] * w[n][cc];
        }
        const float t = wave_sum8(d);
        got = row == j ? t : got;
      }
      if (use) *ge = old + got;
      if constexpr (ONE) break;
    }
  }
#pragma unroll
  for (int cc = 0; cc < NC; ++cc)
    if (lc.live[cc]) gsum[s * ldgs + lc.col[cc]] = acc[cc];
}

RowWeight make_weight(const float* w, int64_t ldw, const int32_t* i1, const int32_t* i2, int64_t ld_idx) {
  return RowWeight{w, ldw, i1, i2, ld_idx};
}

// launch of KERNEL<NC> with NC = ceil(channels / 64) (channels <= 256)
#define TB_LAUNCH_NC(KERNEL, CHANNELS, GRID, ...)                                              \
  do {                                                                                        \
    switch (fmd_cdiv((CHANNELS), 64)) {                                                       \
      case 1: hipLaunchKernelGGL(KERNEL<1>, GRID, dim3(256), 0, stream, __VA_ARGS__); break; \
      case 2: hipLaunchKernelGGL(KERNEL<2>, GRID, dim3(256), 0, stream, __VA_ARGS__); break; \
      case 3: hipLaunchKernelGGL(KERNEL<3>, GRID, dim3(256), 0, stream, __VA_ARGS__); break; \
      default: hipLaunchKernelGGL(KERNEL<4>, GRID, dim3(256), 0, stream, __VA_ARGS__); break; \
    }                                                                                         \
  } while (0)

#define TB_LAUNCH_NC2(KERNEL, FLAG, CHANNELS, GRID, ...)                                              \
  do {                                                                                                \
    switch (fmd_cdiv((CHANNELS), 64)) {                                                               \
      case 1: hipLaunchKernelGGL((KERNEL<1, FLAG>), GRID, dim3(256), 0, stream, __VA_ARGS__); break;  \
      case 2: hipLaunchKernelGGL((KERNEL<2, FLAG>), GRID, dim3(256), 0, stream, __VA_ARGS__); break;  \
      case 3: hipLaunchKernelGGL((KERNEL<3, FLAG>), GRID, dim3(256), 0, stream, __VA_ARGS__); break;  \
      default: hipLaunchKernelGGL((KERNEL<4, FLAG>), GRID, dim3(256), 0, stream, __VA_ARGS__); break; \
    }                                                                                                 \
  } while (0)

}  // namespace

extern "C" {

int fmd_tb_bond_envelope_f32(float* geo, const uint8_t* short_flags, const int64_t* n_edges, int64_t e_cap, float rb,
                             hipStream_t stream) {
  FMD_REQUIRE(e_cap >= 0 && rb > 0.f);
  if (e_cap == 0) return FMD_OK;
  FMD_REQUIRE(geo && short_flags && n_edges);
  hipLaunchKernelGGL(tb_envelope_kernel, dim3((unsigned)fmd_cdiv(e_cap, 256)), dim3(256), 0, stream, geo, short_flags,
                     n_edges, e_cap, rb);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_gated_sum_f32(const float* z, int64_t ldz, int64_t rows, int32_t channels, const float* w, int64_t ldw,
                         const int32_t* index1, const int32_t* index2, int64_t ld_index, const int64_t* offsets,
                         int64_t n_segments, float scale, float* out, int64_t ldo, int32_t accumulate,
                         hipStream_t stream) {
  FMD_REQUIRE(rows >= 0 && n_segments >= 0 && channels > 0 && channels <= 256 && ldz >= channels &&
              ldo >= channels && (index1 || !index2));
  if (n_segments == 0) return FMD_OK;
  FMD_REQUIRE(z && w && offsets && out);
  TB_LAUNCH_NC(tb_gated_sum_kernel, channels, dim3((unsigned)fmd_cdiv(n_segments, 4)), z, ldz, rows, channels,
               make_weight(w, ldw, index1, index2, ld_index), offsets, n_segments, scale, out, ldo, accumulate);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_gated_sum_bwd_f32(const float* gout, int64_t ldg, const float* z, int64_t ldz, int64_t rows,
                             int32_t channels, const float* w, int64_t ldw, const int32_t* index1,
                             const int32_t* index2, int64_t ld_index, const int64_t* offsets, int64_t n_segments,
                             float scale, float* gz, int64_t ldgz, float* gsum, int64_t ldgs, float* gw, int64_t ldgw,
                             int32_t accumulate_gw, hipStream_t stream) {
  FMD_REQUIRE(rows >= 0 && n_segments >= 0 && channels > 0 && channels <= 256 && ldz >= channels &&
              ldgz >= channels && (index1 || !index2));
  if (rows == 0 && n_segments == 0) return FMD_OK;
  FMD_REQUIRE(gout && z && w && offsets && gz);
  FMD_REQUIRE(!gsum || ldgs >= channels);
  FMD_REQUIRE(!gw || ldgw >= (index2 ? 2 : 1));
  const int64_t seg_blocks = fmd_cdiv(n_segments, 4);
  int64_t tail_blocks = fmd_cdiv(rows, 4);
  tail_blocks = tail_blocks < 1 ? 1 : (tail_blocks > 512 ? 512 : tail_blocks);
  TB_LAUNCH_NC(tb_gated_sum_bwd_kernel, channels, dim3((unsigned)(seg_blocks + tail_blocks)), gout, ldg, z, ldz, rows,
               channels, make_weight(w, ldw, index1, index2, ld_index), offsets, n_segments, scale, gz, ldgz, gsum,
               ldgs, gw, ldgw, accumulate_gw, seg_blocks);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_bond_update_f32(const float* u, const float* v, int64_t ldu, const float* h, int64_t ldh, const float* aw,
                           int64_t lda, int32_t channels, const float* geo, const int64_t* short_offsets,
                           const int32_t* bond_rows, const int64_t* edge_triplet_offsets, const int32_t* line_graph,
                           int64_t n_atoms, int64_t t_cap, float scale, float* z3, int64_t ldz, float* eps, int64_t lde,
                           hipStream_t stream) {
  FMD_REQUIRE(n_atoms >= 0 && t_cap >= 0 && channels > 0 && channels <= 256 && ldz >= channels && lde >= channels);
  FMD_REQUIRE(ldu >= channels && ldh >= channels && lda >= channels);
  if (n_atoms == 0 || t_cap == 0) return FMD_OK;
  FMD_REQUIRE(u && v && h && aw && z3 && geo && short_offsets && bond_rows && edge_triplet_offsets && line_graph && eps);
  LineCsr lc{short_offsets, bond_rows, edge_triplet_offsets, nullptr, line_graph, nullptr, n_atoms, t_cap};
  TB_LAUNCH_NC(tb_bond_sum_kernel, channels, dim3(kStrideBlocks), lc, z3, ldz, channels,
               (TripletTerms{u, v, h, aw, ldu, ldh, lda}), geo, scale, eps, lde);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_bond_init_f32(const float* ef, int32_t n_basis, const float* m, int32_t channels,
                         const int64_t* short_offsets, const int32_t* bond_rows, const uint8_t* overflow,
                         int64_t n_atoms, int64_t e_cap, float* out, int64_t ldo, hipStream_t stream) {
  FMD_REQUIRE(n_atoms >= 0 && e_cap >= 0 && channels > 0 && n_basis > 0 && ldo >= 4 * (int64_t)channels);
  if (n_atoms == 0 || e_cap == 0) return FMD_OK;
  FMD_REQUIRE(ef && m && short_offsets && bond_rows && out);
  LineCsr lc{short_offsets, bond_rows, nullptr, nullptr, nullptr, nullptr, n_atoms, 0};
  hipLaunchKernelGGL(tb_bond_init_kernel, dim3(kStrideBlocks), dim3(256), 0, stream, lc, e_cap, ef, n_basis, m, channels,
                     overflow, out, ldo);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_bond_product_f32(const float* a0, int64_t ld0, int32_t k0, const float* a1, int64_t ld1, int32_t k,
                            const float* b, int64_t ldb, int32_t n, const int64_t* short_offsets,
                            const int32_t* bond_rows, const uint8_t* overflow, int64_t n_atoms, int64_t e_cap,
                            float* c, int64_t ldc, int32_t accumulate, hipStream_t stream) {
  FMD_REQUIRE(n_atoms >= 0 && e_cap >= 0 && k0 > 0 && k0 % 32 == 0 && k >= k0 && k % 32 == 0 && n > 0 && n % 64 == 0);
  if (n_atoms == 0 || e_cap == 0) return FMD_OK;
  FMD_REQUIRE(a0 && ld0 >= k0 && b && ldb >= k && c && ldc >= n && short_offsets && bond_rows);
  FMD_REQUIRE(k == k0 || (a1 && ld1 >= k - k0));
  const auto aligned = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  FMD_REQUIRE(aligned(a0) && ld0 % 4 == 0 && aligned(b) && ldb % 4 == 0 && (k == k0 || (aligned(a1) && ld1 % 4 == 0)));
  LineCsr lc{short_offsets, bond_rows, nullptr, nullptr, nullptr, nullptr, n_atoms, 0};
  const BondProduct p{a0, k == k0 ? nullptr : a1, b, c, ld0, ld1, ldb, ldc, k0, k, n, accumulate, overflow};
  if (k <= 64)
    hipLaunchKernelGGL((tb_bond_product_kernel<2>), dim3(2 * kStrideBlocks), dim3(256), 0, stream, lc, e_cap, p);
  else
    hipLaunchKernelGGL((tb_bond_product_kernel<4>), dim3(2 * kStrideBlocks), dim3(256), 0, stream, lc, e_cap, p);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_bond_basis_f32(const float* geps, int64_t ldg, int32_t channels, const float* we, int32_t n_basis,
                          const int64_t* short_offsets, const int32_t* bond_rows, int64_t n_atoms, int64_t e_cap,
                          float* gef, hipStream_t stream) {
  FMD_REQUIRE(n_atoms >= 0 && e_cap >= 0 && channels > 0 && channels <= 256 && n_basis > 0 && ldg >= channels);
  if (n_atoms == 0 || e_cap == 0) return FMD_OK;
  FMD_REQUIRE(geps && we && short_offsets && bond_rows && gef);
  LineCsr lc{short_offsets, bond_rows, nullptr, nullptr, nullptr, nullptr, n_atoms, 0};
  TB_LAUNCH_NC(tb_bond_basis_kernel, channels, dim3(kStrideBlocks), lc, e_cap, geps, ldg, channels, we, n_basis, gef);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_edge_sum_f32(const float* pq, int64_t ldp, const int32_t* edge_index, const float* ef, int32_t n_basis,
                        const float* rt, int32_t channels, const float* geo, const uint8_t* short_flags,
                        const float* bond_part, int64_t ldx, const int64_t* offsets, int64_t n_atoms, int64_t e_cap,
                        float scale, float* z2, float* h, int64_t ldh, hipStream_t stream) {
  FMD_REQUIRE(n_atoms >= 0 && e_cap >= 0 && channels > 0 && channels <= 256 && n_basis > 0 && ldx >= channels);
  FMD_REQUIRE(ldp >= 2 * (int64_t)channels && ldh >= channels);
  if (n_atoms == 0) return FMD_OK;
  FMD_REQUIRE(pq && edge_index && ef && rt && geo && short_flags && bond_part && offsets && z2 && h);
  const EdgeRows er{offsets, e_cap, n_atoms, channels, n_basis, geo, ef, rt};
  const dim3 grid((unsigned)fmd_cdiv(n_atoms, 4));
  if (n_basis <= 8)
    TB_LAUNCH_NC2(tb_edge_sum_kernel, true, channels, grid, er, pq, ldp, edge_index, short_flags, bond_part, ldx, scale,
                  z2, h, ldh);
  else
    TB_LAUNCH_NC2(tb_edge_sum_kernel, false, channels, grid, er, pq, ldp, edge_index, short_flags, bond_part, ldx, scale,
                  z2, h, ldh);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_edge_sum_bwd_f32(const float* gh, int64_t ldg, const float* z2, int32_t n_basis, const float* rt,
                            int32_t channels, const float* geo, const int64_t* offsets, int64_t n_atoms, int64_t e_cap,
                            float scale, float* gz2, float* gsum, int64_t ldgs, float* gfc, float* gef,
                            int32_t accumulate, hipStream_t stream) {
  FMD_REQUIRE(n_atoms >= 0 && e_cap >= 0 && channels > 0 && channels <= 256 && n_basis > 0);
  FMD_REQUIRE(ldg >= channels && ldgs >= channels);
  if (n_atoms == 0) return FMD_OK;
  FMD_REQUIRE(gh && z2 && rt && geo && offsets && gz2 && gsum && gfc && gef);
  const EdgeRows er{offsets, e_cap, n_atoms, channels, n_basis, geo, nullptr, rt};
  const dim3 grid((unsigned)fmd_cdiv(n_atoms, 4));
  if (n_basis <= 8)
    TB_LAUNCH_NC2(tb_edge_sum_bwd_kernel, true, channels, grid, er, gh, ldg, z2, scale, gz2, gsum, ldgs, gfc, gef,
                  accumulate);
  else
    TB_LAUNCH_NC2(tb_edge_sum_bwd_kernel, false, channels, grid, er, gh, ldg, z2, scale, gz2, gsum, ldgs, gfc, gef,
                  accumulate);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_triplet_bwd_f32(const float* geps, int64_t ldg, const float* z3, int64_t ldz, int32_t channels,
                           const float* geo, const int32_t* line_graph, const int64_t* pair_offsets, int64_t n_atoms,
                           int64_t t_cap, float scale, float* gz3, int64_t ldgz, float* gsw, hipStream_t stream) {
  FMD_REQUIRE(n_atoms >= 0 && t_cap >= 0 && channels > 0 && channels <= 256 && ldg >= channels && ldz >= channels &&
              ldgz >= channels);
  if (n_atoms == 0 || t_cap == 0) return FMD_OK;
  FMD_REQUIRE(geps && z3 && geo && line_graph && pair_offsets && gz3 && gsw);
  LineCsr lc{nullptr, nullptr, nullptr, nullptr, line_graph, pair_offsets, n_atoms, t_cap};
  TB_LAUNCH_NC(tb_triplet_bwd_kernel, channels, dim3(kStrideBlocks), lc, geps, ldg, z3, ldz, channels, geo, scale, gz3,
               ldgz, gsw);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_vjp_sums_f32(const float* gz3, int64_t ldz, int32_t channels, const float* gsw,
                        const int64_t* short_offsets, const int32_t* bond_rows, const int64_t* edge_triplet_offsets,
                        const int32_t* second_perm, const int64_t* pair_offsets, int64_t n_atoms, int64_t t_cap,
                        float* guv, int64_t ldg, float* gs, int32_t accumulate_gs, const float* gz2,
                        const int64_t* offsets, const int32_t* reverse, int64_t e_cap, float* s_src, float* s_tri,
                        int64_t lds, hipStream_t stream) {
  FMD_REQUIRE(n_atoms >= 0 && t_cap > 0 && e_cap >= 0 && channels > 0 && channels <= 256 && channels % 64 == 0);
  FMD_REQUIRE(ldz >= channels && ldz % 4 == 0 && ldg >= 2 * (int64_t)channels && lds >= channels && lds % 4 == 0);
  if (n_atoms == 0) return FMD_OK;
  FMD_REQUIRE(gz3 && gsw && short_offsets && bond_rows && edge_triplet_offsets && second_perm && pair_offsets && guv && gs);
  FMD_REQUIRE(offsets && s_src && s_tri && (e_cap == 0 || (gz2 && reverse)));
  const auto aligned = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  FMD_REQUIRE(aligned(gz3) && aligned(gz2) && aligned(s_src) && aligned(s_tri));
  LineCsr lc{short_offsets, bond_rows, edge_triplet_offsets, second_perm, nullptr, pair_offsets, n_atoms, t_cap};
  const NodeSums ns{gz2, offsets, reverse, e_cap, s_src, s_tri, lds};
  const int64_t bond_blocks = kStrideBlocks;
  TB_LAUNCH_NC(tb_vjp_sums_kernel, channels, dim3((unsigned)(bond_blocks + fmd_cdiv(2 * n_atoms, 4))), lc, gz3, ldz,
               channels, gsw, guv, ldg, gs, accumulate_gs, ns, bond_blocks);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_readout_f32(const float* h, int64_t ldh, int32_t channels, const float* wr, const int32_t* elem,
                       const float* e0, int64_t n, float* energy, hipStream_t stream) {
  FMD_REQUIRE(n >= 0 && channels > 0 && ldh >= channels);
  if (n == 0) return FMD_OK;
  FMD_REQUIRE(h && wr && elem && e0 && energy);
  hipLaunchKernelGGL(tb_readout_kernel, dim3((unsigned)fmd_cdiv(n, 4)), dim3(256), 0, stream, h, ldh, channels, wr,
                     elem, e0, n, energy);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_readout_bwd_f32(const float* gE, float sign, const float* wr, int32_t channels, int64_t n, float* gh,
                           int64_t ldgh, hipStream_t stream) {
  FMD_REQUIRE(n >= 0 && channels > 0 && ldgh >= channels);
  if (n == 0) return FMD_OK;
  FMD_REQUIRE(wr && gh);
  hipLaunchKernelGGL(tb_readout_bwd_kernel, dim3((unsigned)fmd_cdiv(n * channels, 256)), dim3(256), 0, stream, gE,
                     sign, wr, channels, n, gh, ldgh);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_geometry_bwd_f32(const float* geo, const float* def, int32_t nb, const float* gef, int64_t ldgef,
                            const float* gu, int64_t ldgu, const float* gfc, const float* gs, const uint8_t* bond_flags,
                            const int64_t* n_edges, int64_t e_cap, float* gvec, hipStream_t stream) {
  FMD_REQUIRE(e_cap >= 0 && nb > 0);
  if (e_cap == 0) return FMD_OK;
  FMD_REQUIRE(geo && def && n_edges && gvec);
  FMD_REQUIRE(!gef || ldgef >= nb);
  FMD_REQUIRE(!gu || ldgu >= 3);
  const RowGrads rg{geo, def, gef, gu, gfc, gs, bond_flags, ldgef, ldgu, nb, false};
  hipLaunchKernelGGL(tb_geometry_bwd_kernel, dim3((unsigned)fmd_cdiv(e_cap, 256)), dim3(256), 0, stream, rg, n_edges,
                     e_cap, gvec);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_tb_edge_forces_f32(const float* geo, const float* def, int32_t nb, const float* gef, int64_t ldgef,
                           const float* gu, int64_t ldgu, const float* gfc, const float* gs, const uint8_t* bond_flags,
                           const int64_t* offsets, const int32_t* reverse, const int64_t* n_edges, int64_t e_cap,
                           int64_t n_atoms, float sign, float* forces, float* gvec, hipStream_t stream) {
  FMD_REQUIRE(n_atoms >= 0 && e_cap >= 0 && nb > 0);
  if (n_atoms == 0) return FMD_OK;
  FMD_REQUIRE(offsets && n_edges && forces && (e_cap == 0 || (geo && def && reverse)));
  FMD_REQUIRE(!gef || ldgef >= nb);
  FMD_REQUIRE(!gu || ldgu >= 3);
  const bool wide = nb == 8 && fmd_wide_rows(def, 8) && (!gef || fmd_wide_rows(gef, ldgef));
  const RowGrads rg{geo, def, gef, gu, gfc, gs, bond_flags, ldgef, ldgu, nb, wide};
  hipLaunchKernelGGL(tb_edge_forces_kernel, dim3((unsigned)fmd_cdiv(n_atoms, 4)), dim3(256), 0, stream, rg, offsets,
                     reverse, n_edges, e_cap, n_atoms, sign, forces, gvec);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

}  // extern "C"
