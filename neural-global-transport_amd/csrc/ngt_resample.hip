// SampleGridLut / SampleGridTransform / LodTransform and their adjoints on
// gfx950, with mip-mapped reads.
//
// Forward kernels: one work-item per output cell, x fastest, 64x4 work-groups
// so a wavefront reads 64 consecutive LUT float4s (coalesced) and writes 64
// consecutive output cells; the 8-tap gathers hit L2/MALL (the whole input of
// the configurations here is cache-resident).  All (batch, camera) pairs go in
// one launch (grid.z = depth x pairs) instead of the reference's per-camera
// launch + device sync loop (resample_grid.cu.cc:712-794).
//
// Backward: a table's positions are arbitrary, so its input gradient is a
// scatter with hardware fp32 atomics, and so is a transform's where it is not
// the gather below; the LUT gradient is a pure gather (data gradient . dy)
// accumulated over the data batch in registers.
//
// Mips: the pyramid of every batch entry is built once per call in the
// workspace (one launch per level, 2x2x2 means in the reference's pairwise
// order z, y, x: resample_grid.cu.cc:58-84).  The exact adjoint scatters into
// per-level gradient buffers and collapses them coarse to fine, each fine
// cell adding 1/8 of its parent (no atomics in the collapse).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "ngt_host.hpp"

namespace ngt {
namespace {

constexpr int kBX = 64, kBY = 4;
constexpr int kMaxMips = 16;

// ----------------------------------------------------------------- mips -----

NGT_HOST_DEVICE_INLINE Dims level_dims(const Dims& d, int m) { return Dims{d.x >> m, d.y >> m, d.z >> m}; }
// A pyramid of n_data grids: level 0 is the caller's buffer (`base`, N
// slices); levels 1..L follow each other in `levels`, level m holding
// [N][dims >> m][C].
struct MipSet {
  float* base;
  float* levels;
  Dims d0;
  int n_data;
  int num_levels;  // L
};

template <int C>
NGT_HOST_DEVICE_INLINE float* level_ptr(const MipSet& s, int n, int m, Dims& dm) {
  dm = level_dims(s.d0, m);
  if (m == 0) return s.base + n * dims_cells(s.d0) * C;
  int64_t off = 0;
  for (int k = 1; k < m; ++k) off += dims_cells(level_dims(s.d0, k));
  return s.levels + (off * s.n_data + n * dims_cells(dm)) * C;
}

// floats of levels 1..L of N grids
int64_t mip_floats(const Dims& d0, int64_t n, int64_t c, int levels) {
  int64_t f = 0;
  for (int m = 1; m <= levels; ++m) f += dims_cells(level_dims(d0, m));
  return f * n * c;
}

size_t align256(size_t b) { return (b + 255) / 256 * 256; }

// Level choice of one sample (Sampler2::sample3D, sampling.hpp:939-1010).
struct MipPick {
  int lf, lc;
  float wc;     // weight of level lc (0 unless two levels are read)
  bool two;     // LINEAR and lc > lf
  bool inside;  // raw + bias strictly inside (0, L): d lod / d raw = 1
};

template <int MM>
NGT_DEVICE MipPick mip_pick(float lod_raw, float bias, int L) {
  const float raw = lod_raw + bias;
  const float lod = fminf(fmaxf(raw, 0.f), static_cast<float>(L));
  MipPick p;
  if constexpr (MM == NGT_MIP_NEAREST) {
    p.lf = min(static_cast<int>(lod + 0.5f), L);
    p.lc = p.lf;
    p.two = false;
    p.wc = 0.f;
  } else {
    p.lf = min(static_cast<int>(lod), L);
    p.lc = min(static_cast<int>(ceilf(lod)), L);
    p.two = p.lc > p.lf;
    p.wc = p.two ? lod - floorf(lod) : 0.f;
  }
  p.inside = raw > 0.f && raw < static_cast<float>(L);
  return p;
}

NGT_DEVICE float level_scale(int m) { return 1.f / static_cast<float>(1 << m); }

template <int C, int FM, int BM>
NGT_DEVICE Vec<C> read_level(const MipSet& s, int n, int m, float px, float py, float pz, float cco) {
  Dims dm;
  const float* g = level_ptr<C>(s, n, m, dm);
  const float sc = level_scale(m);
  return read_filtered<C, FM, BM>(g, dm, px * sc - cco, py * sc - cco, pz * sc - cco);
}

// Mip-mapped read of position p (before the cell-centre offset).  The levels
// are visited one by one, those that no lane of the wavefront reads skipped:
// a level's address and extents are then scalar (a level of its own per lane
// walks the pyramid's offsets in 64-bit vector arithmetic, twice).
template <int C, int FM, int BM, int MM>
NGT_DEVICE Vec<C> read_mip(const MipSet& s, int n, float px, float py, float pz, float lod_raw, float bias,
                           float cco) {
  const MipPick k = mip_pick<MM>(lod_raw, bias, s.num_levels);
  Vec<C> rf = vzero<C>(), rc = vzero<C>();
  for (int m = 0; m <= s.num_levels; ++m) {
    const bool low = k.lf == m, high = MM == NGT_MIP_LINEAR && k.two && k.lc == m;
    if (low || high) {
      const Vec<C> v = read_level<C, FM, BM>(s, n, m, px, py, pz, cco);
#pragma unroll
      for (int i = 0; i < C; ++i) {
        rf.v[i] = low ? v.v[i] : rf.v[i];
        rc.v[i] = high ? v.v[i] : rc.v[i];
      }
    }
  }
  if constexpr (MM == NGT_MIP_LINEAR) {
    if (k.two) rf = vlerp(rf, rc, k.wc);
  }
  return rf;
}

template <int C, int FM, int BM>
NGT_DEVICE void scatter_level(const MipSet& data, const MipSet& grad, int n, int m, float px, float py, float pz,
                              float cco, const Vec<C>& val) {
  Dims dm;
  const float* src = level_ptr<C>(data, n, m, dm);
  float* g = level_ptr<C>(grad, n, m, dm);
  const float sc = level_scale(m);
  scatter_filtered<C, FM, BM>(src, g, dm, px * sc - cco, py * sc - cco, pz * sc - cco, val);
}

// Level m+1 of n_data grids from level m: each cell the mean of its 2x2x2
// children, averaged along z, then y, then x.
template <int C>
__global__ __launch_bounds__(256) void mip_down_kernel(const float* __restrict__ fine, Dims df,
                                                       float* __restrict__ coarse, Dims dc, int n_data) {
  const int64_t cells = dims_cells(dc);
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= cells * n_data) return;
  const int n = static_cast<int>(i / cells);
  int64_t r = i - n * cells;
  const int x = static_cast<int>(r % dc.x);
  r /= dc.x;
  const int y = static_cast<int>(r % dc.y);
  const int z = static_cast<int>(r / dc.y);
  const float* f = fine + n * dims_cells(df) * C;
  Vec<C> v[2][2][2];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int a = 0; a < 2; ++a) v[c][b][a] = vload<C>(f + cell_offset(df, 2 * x + a, 2 * y + b, 2 * z + c) * C);
  Vec<C> out;
#pragma unroll
  for (int k = 0; k < C; ++k) {
    float yx[2][2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int a = 0; a < 2; ++a) yx[b][a] = (v[0][b][a].v[k] + v[1][b][a].v[k]) * 0.5f;
    const float x0 = (yx[0][0] + yx[1][0]) * 0.5f;
    const float x1 = (yx[0][1] + yx[1][1]) * 0.5f;
    out.v[k] = (x0 + x1) * 0.5f;
  }
  vstore<C>(coarse + (n * cells + cell_offset(dc, x, y, z)) * C, out);
}

// Adjoint of one mip_down: every fine cell of the 2*dims_coarse region adds
// 1/8 of its parent's gradient.
template <int C>
__global__ __launch_bounds__(256) void mip_collapse_kernel(const float* __restrict__ coarse, Dims dc,
                                                           float* __restrict__ fine, Dims df, int n_data) {
  const Dims dr{2 * dc.x, 2 * dc.y, 2 * dc.z};
  const int64_t cells = dims_cells(dr);
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= cells * n_data) return;
  const int n = static_cast<int>(i / cells);
  int64_t r = i - n * cells;
  const int x = static_cast<int>(r % dr.x);
  r /= dr.x;
  const int y = static_cast<int>(r % dr.y);
  const int z = static_cast<int>(r / dr.y);
  const Vec<C> p = vload<C>(coarse + (n * dims_cells(dc) + cell_offset(dc, x >> 1, y >> 1, z >> 1)) * C);
  float* o = fine + (n * dims_cells(df) + cell_offset(df, x, y, z)) * C;
  Vec<C> v = vload<C>(o);
#pragma unroll
  for (int k = 0; k < C; ++k) v.v[k] += 0.125f * p.v[k];
  vstore<C>(o, v);
}

template <int C>
void launch_mip_generate(const MipSet& s, hipStream_t st) {
  for (int m = 0; m < s.num_levels; ++m) {
    Dims df, dc;
    const float* f = level_ptr<C>(s, 0, m, df);
    float* c = level_ptr<C>(s, 0, m + 1, dc);
    const int64_t n = dims_cells(dc) * s.n_data;
    hipLaunchKernelGGL((mip_down_kernel<C>), dim3(blocks_for(n, 256)), dim3(256), 0, st, f, df, c, dc, s.n_data);
  }
}

template <int C>
void launch_mip_collapse(const MipSet& g, hipStream_t st) {
  for (int m = g.num_levels; m >= 1; --m) {
    Dims df, dc;
    float* f = level_ptr<C>(g, 0, m - 1, df);
    const float* c = level_ptr<C>(g, 0, m, dc);
    const int64_t n = 8 * dims_cells(dc) * g.n_data;
    hipLaunchKernelGGL((mip_collapse_kernel<C>), dim3(blocks_for(n, 256)), dim3(256), 0, st, c, dc, f, df, g.n_data);
  }
}

// ------------------------------------------------------------------ LUT -----

struct LutArgs {
  const float* input;
  Dims din;
  const float* lut;
  Dims dout;
  int n_data, n_cams, separate;
  float cco;
  int relative, normalized;
  float mip_bias;
};

// Sample position (before the cell-centre offset) and raw LoD of one LUT cell
// (resample_grid.cu.cc:610-618).
NGT_DEVICE void lut_position(const LutArgs& a, int v, int x, int y, int z, float& px, float& py, float& pz,
                             float& lod) {
  const float4 l = *reinterpret_cast<const float4*>(a.lut + (cell_offset(a.dout, x, y, z) + static_cast<int64_t>(v) * a.dout.x * a.dout.y * a.dout.z) * 4);
  px = l.x; py = l.y; pz = l.z; lod = l.w;
  if (a.normalized) {
    px *= static_cast<float>(a.dout.x); py *= static_cast<float>(a.dout.y); pz *= static_cast<float>(a.dout.z);
  }
  if (a.relative) {
    px += static_cast<float>(x); py += static_cast<float>(y); pz += static_cast<float>(z);
  }
}

template <int C, int FM, int BM, int MM>
__global__ __launch_bounds__(256) void lut_fwd_kernel(LutArgs a, MipSet mips, float* __restrict__ out) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  const int z = blockIdx.z % a.dout.z;
  const int pair = blockIdx.z / a.dout.z;
  if (x >= a.dout.x || y >= a.dout.y) return;
  int n, v;
  if (a.separate) { n = pair / a.n_cams; v = pair % a.n_cams; }
  else { n = pair; v = pair; }
  float px, py, pz, lod;
  lut_position(a, v, x, y, z, px, py, pz, lod);
  Vec<C> r;
  if constexpr (MM == NGT_MIP_NONE) {
    const int64_t in_slice = static_cast<int64_t>(a.din.x) * a.din.y * a.din.z * C;
    r = read_filtered<C, FM, BM>(a.input + n * in_slice, a.din, px - a.cco, py - a.cco, pz - a.cco);
  } else {
    r = read_mip<C, FM, BM, MM>(mips, n, px, py, pz, lod, a.mip_bias, a.cco);
  }
  const int64_t out_cells = static_cast<int64_t>(a.dout.x) * a.dout.y * a.dout.z;
  vstore<C>(out + (static_cast<int64_t>(pair) * out_cells + cell_offset(a.dout, x, y, z)) * C, r);
}

// -------------------------------------------------- scatter through LDS -----
// The LINEAR table adjoint works on 3-D tiles of output cells, 256 work-items
// of S cells each.  Adding 8 corners per sample to the gradient is bound by the
// rate of scattered global atomics (21 to 85 G/s here; coalesced ones reach 327
// G/s).  Neighbouring cells sample neighbouring places, so a tile's corners are
// added to fp64 sums in LDS over their bounding box, and the box is added to
// the gradient once, in rows: one global atomic per touched value.  A tile
// whose box does not fit, or that holds a position that is no number, adds its
// corners to the gradient directly.
// A 128^3 table of one channel: 164 us -> 36.7 us, 64^3: 13.2 -> 8.9 us.  Of
// the tiles at one channel 16 x 8 x 4 is the fastest: 16 x 8 x 8 takes 44 (11.6)
// us, 8 x 8 x 8 44 (9.9), 8 x 8 x 4 46 (10.7).
template <int C>
struct ScatterTile {
  static constexpr int S = C == 4 ? 1 : 2;
  static constexpr int X = C == 4 ? 8 : 16, Y = 8, Z = 4;
  static constexpr int kValues = C == 4 ? 6144 : 4096;  // 48 and 32 KB, with the box: three and four work-groups per CU

  static dim3 block() { return dim3(X, Y, Z / S); }
  // Tiles along x and y, and along z for every slot: no axis has more
  // work-groups than one work-item per cell would need.
  static dim3 grid(const Dims& d, int slots) {
    return dim3((d.x + X - 1) / X, (d.y + Y - 1) / Y, (d.z + Z - 1) / Z * slots);
  }
};

NGT_DEVICE int flat_thread() { return (threadIdx.z * blockDim.y + threadIdx.y) * blockDim.x + threadIdx.x; }

// Smallest value of the wavefront, in lane 63: minima over rows of 16 lanes,
// then across the rows, as DPP operands of the minimum (a shuffle is an LDS
// operation).
template <int CTRL, int ROWS>
NGT_DEVICE int dpp_min(int v) {
  return min(v, __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xf, false));
}
NGT_DEVICE int wave_min(int v) {
  v = dpp_min<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
  v = dpp_min<0x112, 0xf>(v);
  v = dpp_min<0x114, 0xf>(v);
  v = dpp_min<0x118, 0xf>(v);
  v = dpp_min<0x142, 0xa>(v);  // row_bcast 15 into rows 1 and 3
  return dpp_min<0x143, 0xc>(v);  // row_bcast 31 into rows 2 and 3
}

struct ScatterShared {
  int box[4][6];
  int ok[4];
};

// Scatters val[s] to the corners of q[s] (where live[s]; for BORDER only
// samples inside) into g.  Called by the whole work-group; the LDS is free again
// when it returns.
template <int C, int BM>
NGT_DEVICE void tile_scatter(double* sums, ScatterShared& sh, float* __restrict__ g, const Dims& d,
                             const float (&qx)[ScatterTile<C>::S], const float (&qy)[ScatterTile<C>::S],
                             const float (&qz)[ScatterTile<C>::S], const Vec<C> (&val)[ScatterTile<C>::S],
                             const bool (&live)[ScatterTile<C>::S]) {
  constexpr int S = ScatterTile<C>::S;
  const int tid = flat_thread();
  // floor and ceil cells (clamped for CLAMP, not wrapped for WRAP) of the
  // samples that are read
  int lo[S][3], step[S][3];
  int mn[3] = {1 << 30, 1 << 30, 1 << 30}, mx[3] = {-(1 << 30), -(1 << 30), -(1 << 30)};
  bool ok = true;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const float q[3] = {qx[s], qy[s], qz[s]};
    const int dims[3] = {d.x, d.y, d.z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const bool number = fabsf(q[k]) < 1.0e8f;
      ok = ok & (number | !live[s]);
      const float f = number ? floorf(q[k]) : 0.f;
      int i0 = static_cast<int>(f), i1 = i0 + (q[k] != f ? 1 : 0);
      if constexpr (BM == CLAMP) {
        i0 = min(max(i0, 0), dims[k] - 1);
        i1 = min(max(i1, 0), dims[k] - 1);
      }
      lo[s][k] = i0;
      step[s][k] = i1 - i0;
      if (live[s]) {
        mn[k] = min(mn[k], i0);
        mx[k] = max(mx[k], i1);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    mn[k] = wave_min(mn[k]);
    mx[k] = -wave_min(-mx[k]);
  }
  const bool wave_ok = __all(ok);
  if ((tid & 63) == 63) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      sh.box[tid >> 6][k] = mn[k];
      sh.box[tid >> 6][3 + k] = mx[k];
    }
    sh.ok[tid >> 6] = wave_ok;
  }
  __syncthreads();
  int ext[3];
  bool fits = true;
#pragma unroll
  for (int w = 0; w < 4; ++w) fits = fits && sh.ok[w];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    mn[k] = min(min(sh.box[0][k], sh.box[1][k]), min(sh.box[2][k], sh.box[3][k]));
    mx[k] = max(max(sh.box[0][3 + k], sh.box[1][3 + k]), max(sh.box[2][3 + k], sh.box[3][3 + k]));
    ext[k] = max(0, mx[k] - mn[k] + 1);
    fits = fits && ext[k] <= ScatterTile<C>::kValues;
  }
  const int64_t volume = static_cast<int64_t>(ext[0]) * ext[1] * ext[2];
  if (!fits || volume * C > ScatterTile<C>::kValues) {  // uniform
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (live[s]) scatter_linear<C, BM, false>(g, d, qx[s], qy[s], qz[s], val[s]);
    __syncthreads();  // sh is written again by the next call
    return;
  }
  const int n = static_cast<int>(volume) * C;
  for (int i = tid; i < n; i += 256) sums[i] = 0.0;
  __syncthreads();
  const int rx = C, ry = ext[0] * C, rz = ext[0] * ext[1] * C;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    if (!live[s]) continue;
    const float wx = qx[s] - floorf(qx[s]), wy = qy[s] - floorf(qy[s]), wz = qz[s] - floorf(qz[s]);
    const float fw[2][3] = {{1.f - wx, 1.f - wy, 1.f - wz}, {wx, wy, wz}};
    double* const t = sums + (lo[s][0] - mn[0]) * rx + (lo[s][1] - mn[1]) * ry + (lo[s][2] - mn[2]) * rz;
    const int sx = step[s][0] * rx, sy = step[s][1] * ry, sz = step[s][2] * rz;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int bx = k & 1, by = (k >> 1) & 1, bz = k >> 2;
      const float w = fw[bx][0] * fw[by][1] * fw[bz][2];
      double* const p = t + (bx ? sx : 0) + (by ? sy : 0) + (bz ? sz : 0);
#pragma unroll
      for (int j = 0; j < C; ++j) lds_add(p + j, val[s].v[j] * w);
    }
  }
  __syncthreads();
  // the box in rows of ext[0] * C values
  const int len = ext[0] * C;
  const float inv_len = 1.f / static_cast<float>(max(len, 1)), inv_ext = 1.f / static_cast<float>(max(ext[1], 1));
  for (int i = tid; i < n; i += 256) {
    const float v = static_cast<float>(sums[i]);
    if (v == 0.f) continue;
    // exact: i < kValues, so the estimate is off by less than one half
    const int row = static_cast<int>((static_cast<float>(i) + 0.5f) * inv_len), c = i - row * len;
    const int lz = static_cast<int>((static_cast<float>(row) + 0.5f) * inv_ext);
    int x = mn[0] + c / C, y = mn[1] + row - lz * ext[1], z = mn[2] + lz;
    if constexpr (BM == BORDER) {
      if (x < 0 || x >= d.x || y < 0 || y >= d.y || z < 0 || z >= d.z) continue;
    } else if constexpr (BM == WRAP) {
      x = wrap_index(x, d.x); y = wrap_index(y, d.y); z = wrap_index(z, d.z);
    }
    atomic_add(g + cell_offset(d, x, y, z) * C + c % C, v);
  }
  __syncthreads();
}

// Exact adjoint of the LINEAR table read, with mips where MM is not NONE: the
// input gradient through tile_scatter (level by level), the LUT gradient in
// registers over the data entries that use this camera.
template <int C, int BM, int MM>
__global__ __launch_bounds__(256) void lut_bwd_tile_kernel(LutArgs a, MipSet data, MipSet grad,
                                                           const float* __restrict__ out_grad,
                                                           float* __restrict__ lut_grad) {
  using T = ScatterTile<C>;
  constexpr int S = T::S;
  __shared__ double sums[T::kValues];
  __shared__ ScatterShared sh;
  const int tiles_z = (a.dout.z + T::Z - 1) / T::Z;
  const int v = blockIdx.z / tiles_z, tz = blockIdx.z % tiles_z;
  const int64_t out_cells = dims_cells(a.dout);
  int64_t cell[S];
  bool on[S];
  float px[S], py[S], pz[S];
  MipPick k[S];
  float gx[S], gy[S], gz[S], gl[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    int x = blockIdx.x * T::X + threadIdx.x, y = blockIdx.y * T::Y + threadIdx.y;
    int z = tz * T::Z + static_cast<int>(threadIdx.z) * S + s;
    on[s] = x < a.dout.x && y < a.dout.y && z < a.dout.z;
    x = min(x, a.dout.x - 1); y = min(y, a.dout.y - 1); z = min(z, a.dout.z - 1);
    cell[s] = cell_offset(a.dout, x, y, z);
    float lod;
    lut_position(a, v, x, y, z, px[s], py[s], pz[s], lod);
    if constexpr (MM != NGT_MIP_NONE) k[s] = mip_pick<MM>(lod, a.mip_bias, data.num_levels);
    gx[s] = gy[s] = gz[s] = gl[s] = 0.f;
  }
  const int n_begin = a.separate ? 0 : v;
  const int n_end = a.separate ? a.n_data : v + 1;
  for (int n = n_begin; n < n_end; ++n) {
    const int slot = a.separate ? n * a.n_cams + v : n;
    Vec<C> dy[S];
#pragma unroll
    for (int s = 0; s < S; ++s) dy[s] = vload<C>(out_grad + (static_cast<int64_t>(slot) * out_cells + cell[s]) * C);
    Vec<C> low[S];  // the finer level's value, for the derivative of the level lerp
    for (int m = 0; m <= grad.num_levels; ++m) {
      Dims dm;
      const float* const src = level_ptr<C>(data, n, m, dm);
      float* const g = level_ptr<C>(grad, n, m, dm);
      const float sc = level_scale(m);
      float qx[S], qy[S], qz[S];
      Vec<C> val[S];
      bool here[S];
      bool some = false;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        here[s] = on[s];
        float w = 1.f;
        bool fine = true;
        if constexpr (MM != NGT_MIP_NONE) {
          fine = k[s].lf == m;
          here[s] = on[s] && (fine || (k[s].two && k[s].lc == m));
          w = fine ? 1.f - k[s].wc : k[s].wc;
        }
        qx[s] = px[s] * sc - a.cco; qy[s] = py[s] * sc - a.cco; qz[s] = pz[s] * sc - a.cco;
        val[s] = vscale(dy[s], w);
        if (here[s]) {
          if constexpr (BM == BORDER) here[s] = inside_border(dm, qx[s], qy[s], qz[s]);
          Vec<C> r = {}, dx = {}, dyy = {}, dz = {};
          if (here[s]) r = read_linear_gradient<C, BM>(src, dm, qx[s], qy[s], qz[s], dx, dyy, dz);
          gx[s] += w * sc * vdot(dy[s], dx); gy[s] += w * sc * vdot(dy[s], dyy); gz[s] += w * sc * vdot(dy[s], dz);
          if constexpr (MM == NGT_MIP_LINEAR) {
            if (fine) low[s] = r;
            else if (k[s].inside) gl[s] += vdot(dy[s], vsub(r, low[s]));
          }
        }
        some = some || here[s];
      }
      if (MM == NGT_MIP_NONE || __syncthreads_or(some)) tile_scatter<C, BM>(sums, sh, g, dm, qx, qy, qz, val, here);
    }
  }
#pragma unroll
  for (int s = 0; s < S; ++s) {
    if (!on[s]) continue;
    if (a.normalized) {
      gx[s] *= static_cast<float>(a.dout.x); gy[s] *= static_cast<float>(a.dout.y); gz[s] *= static_cast<float>(a.dout.z);
    }
    *reinterpret_cast<float4*>(lut_grad + (static_cast<int64_t>(v) * out_cells + cell[s]) * 4) =
        make_float4(gx[s], gy[s], gz[s], gl[s]);
  }
}

// The table adjoint without mips of NEAREST / MIN / MAX, whose LUT gradient is
// 0, and the reference's (REF: FM is LINEAR where it has a LUT gradient).  One
// work-item per (camera slot, output cell); loops over the data entries that
// use this camera.
template <int C, int FM, int BM, bool REF>
__global__ __launch_bounds__(256) void lut_bwd_kernel(LutArgs a, const float* __restrict__ out_grad,
                                                      float* __restrict__ in_grad, float* __restrict__ lut_grad,
                                                      uint32_t* __restrict__ hits) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  const int z = blockIdx.z % a.dout.z;
  const int v = blockIdx.z / a.dout.z;
  if (x >= a.dout.x || y >= a.dout.y) return;
  float px, py, pz, lod;
  lut_position(a, v, x, y, z, px, py, pz, lod);
  px -= a.cco; py -= a.cco; pz -= a.cco;
  const int64_t in_cells = static_cast<int64_t>(a.din.x) * a.din.y * a.din.z;
  const int64_t out_cells = static_cast<int64_t>(a.dout.x) * a.dout.y * a.dout.z;
  const int64_t cell = cell_offset(a.dout, x, y, z);
  float g0 = 0.f, g1 = 0.f, g2 = 0.f;
  const int n_begin = a.separate ? 0 : v;
  const int n_end = a.separate ? a.n_data : v + 1;
  for (int n = n_begin; n < n_end; ++n) {
    const int slot = a.separate ? n * a.n_cams + v : n;
    const Vec<C> dy = vload<C>(out_grad + (static_cast<int64_t>(slot) * out_cells + cell) * C);
    const float* src = a.input + n * in_cells * C;
    if constexpr (REF) {
      if constexpr (FM == LINEAR) {  // written per camera, the last batch entry wins
        Vec<C> dx, dyy, dz;
        read_gradient<C, BM>(src, a.din, px, py, pz, dx, dyy, dz);
        g0 = vdot(dy, dx); g1 = vdot(dy, dyy); g2 = vdot(dy, dz);
      }
      scatter_linear<C, BM, true>(in_grad + n * in_cells * C, a.din, px, py, pz, dy, hits + n * in_cells);
    } else {
      scatter_filtered<C, FM, BM>(src, in_grad + n * in_cells * C, a.din, px, py, pz, dy);
    }
  }
  *reinterpret_cast<float4*>(lut_grad + (static_cast<int64_t>(v) * out_cells + cell) * 4) = make_float4(g0, g1, g2, 0.f);
}

// Exact adjoint of the mip-mapped NEAREST / MIN / MAX table read: scatter into
// the levels read; the LUT gradient is, in w, the derivative of the level lerp.
template <int C, int FM, int BM, int MM>
__global__ __launch_bounds__(256) void lut_bwd_mip_kernel(LutArgs a, MipSet data, MipSet grad,
                                                          const float* __restrict__ out_grad,
                                                          float* __restrict__ lut_grad) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  const int z = blockIdx.z % a.dout.z;
  const int v = blockIdx.z / a.dout.z;
  if (x >= a.dout.x || y >= a.dout.y) return;
  float px, py, pz, lod_raw;
  lut_position(a, v, x, y, z, px, py, pz, lod_raw);
  const MipPick k = mip_pick<MM>(lod_raw, a.mip_bias, data.num_levels);
  const float wf = 1.f - k.wc;
  const int64_t out_cells = static_cast<int64_t>(a.dout.x) * a.dout.y * a.dout.z;
  const int64_t cell = cell_offset(a.dout, x, y, z);
  float gl = 0.f;
  const int n_begin = a.separate ? 0 : v;
  const int n_end = a.separate ? a.n_data : v + 1;
  for (int n = n_begin; n < n_end; ++n) {
    const int slot = a.separate ? n * a.n_cams + v : n;
    const Vec<C> dy = vload<C>(out_grad + (static_cast<int64_t>(slot) * out_cells + cell) * C);
    scatter_level<C, FM, BM>(data, grad, n, k.lf, px, py, pz, a.cco, vscale(dy, wf));
    if (k.two) scatter_level<C, FM, BM>(data, grad, n, k.lc, px, py, pz, a.cco, vscale(dy, k.wc));
    if constexpr (MM == NGT_MIP_LINEAR) {
      if (k.two && k.inside) {
        const Vec<C> vf = read_level<C, FM, BM>(data, n, k.lf, px, py, pz, a.cco);
        const Vec<C> vc = read_level<C, FM, BM>(data, n, k.lc, px, py, pz, a.cco);
        gl += vdot(dy, vsub(vc, vf));
      }
    }
  }
  *reinterpret_cast<float4*>(lut_grad + (static_cast<int64_t>(v) * out_cells + cell) * 4) = make_float4(0.f, 0.f, 0.f, gl);
}

// grad /= hits where hits > 0 (resample_grid.cu.cc:1133-1151).
template <int C>
__global__ __launch_bounds__(256) void normalize_by_count_kernel(float* __restrict__ g, const uint32_t* __restrict__ hits,
                                                                 int64_t cells) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= cells) return;
  const uint32_t h = hits[i];
  if (h > 0u) {
    const float w = 1.0f / static_cast<float>(h);
    Vec<C> d = vload<C>(g + i * C);
    vstore<C>(g + i * C, vscale(d, w));
  }
}

// ----------------------------------------------------------- transform ------

struct XformArgs {
  const float* input;
  Dims din;
  Dims dout;
  float out_inv_x, out_inv_y, out_inv_z;
  int coord_mode;
  float mip_bias;
};

// samplePos3D<CM, false> at index coordinates (cell index + 0.5).
NGT_DEVICE void xform_pos(const XformArgs& a, const CamParams& cp, float ix, float iy, float iz, float& px, float& py,
                          float& pz) {
  switch (a.coord_mode) {
    case NGT_COORD_TRANSFORM:
      idx_to_os(cp, ix, iy, iz, a.out_inv_x, a.out_inv_y, a.out_inv_z, px, py, pz);
      break;
    case NGT_COORD_TRANSFORM_REVERSE:
      os_to_idx(cp, ix, iy, iz, static_cast<float>(a.din.x), static_cast<float>(a.din.y), static_cast<float>(a.din.z),
                px, py, pz);
      break;
    case NGT_COORD_TRANSFORM_LINDEPTH_REVERSE:
      os_to_idx_lindepth(cp, ix, iy, iz, static_cast<float>(a.din.x), static_cast<float>(a.din.y),
                         static_cast<float>(a.din.z), px, py, pz);
      break;
    default:
      idx_to_os_lindepth(cp, ix, iy, iz, a.out_inv_x, a.out_inv_y, a.out_inv_z, px, py, pz);
      break;
  }
}

NGT_DEVICE bool forward_mode(int cm) { return cm == NGT_COORD_TRANSFORM || cm == NGT_COORD_TRANSFORM_LINDEPTH; }

NGT_DEVICE float log2_lod(float l0, float l1, float l2) { return fmaxf(0.f, log2f(fmaxf(l0, fmaxf(l1, l2)))); }

// Raw LoD of samplePos3D<CM, true> (sampling.hpp:158-228): forward
// differences p - p(idx + e); per object-space axis lengths in the forward
// modes, per difference vector in the reverse modes.
NGT_DEVICE float xform_lod(const XformArgs& a, const CamParams& cp, float ix, float iy, float iz, float px, float py,
                           float pz) {
  float d[3][3];
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    float qx, qy, qz;
    xform_pos(a, cp, ix + (e == 0 ? 1.f : 0.f), iy + (e == 1 ? 1.f : 0.f), iz + (e == 2 ? 1.f : 0.f), qx, qy, qz);
    d[e][0] = px - qx; d[e][1] = py - qy; d[e][2] = pz - qz;
  }
  float l[3];
  if (forward_mode(a.coord_mode)) {
#pragma unroll
    for (int k = 0; k < 3; ++k) l[k] = sqrtf(d[0][k] * d[0][k] + d[1][k] * d[1][k] + d[2][k] * d[2][k]);
  } else {
#pragma unroll
    for (int e = 0; e < 3; ++e) l[e] = sqrtf(d[e][0] * d[e][0] + d[e][1] * d[e][1] + d[e][2] * d[e][2]);
  }
  return log2_lod(l[0], l[1], l[2]);
}

// Whether position p may be valid under BORDER at any level: level m is read
// at q = p / 2^m - 0.5 (rounded), valid for 0 <= q + 0.5 < dims >> m, and
// (dims >> m) << m <= dims; one cell of slack covers the roundings.
NGT_DEVICE bool xform_inside(const Dims& d, float px, float py, float pz) {
  return (px > -1.f) & (px < static_cast<float>(d.x) + 1.f) & (py > -1.f) & (py < static_cast<float>(d.y) + 1.f) &
         (pz > -1.f) & (pz < static_cast<float>(d.z) + 1.f);
}

template <int C, int FM, int BM, int MM>
__global__ __launch_bounds__(256) void xform_fwd_kernel(XformArgs a, CamBatch cb, MipSet mips,
                                                        float* __restrict__ out) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  const int z = blockIdx.z % a.dout.z;
  const int ci = blockIdx.z / a.dout.z;
  if (x >= a.dout.x || y >= a.dout.y) return;
  const CamParams& cp = cb.cam[ci];
  const float ix = static_cast<float>(x) + 0.5f, iy = static_cast<float>(y) + 0.5f, iz = static_cast<float>(z) + 0.5f;
  float px, py, pz;
  xform_pos(a, cp, ix, iy, iz, px, py, pz);
  const int64_t in_slice = static_cast<int64_t>(a.din.x) * a.din.y * a.din.z * C;
  Vec<C> r;
  if constexpr (BM == WRAP) {
    r = vzero<C>();  // Sampler2 has no WRAP path (sampling.hpp:802-826)
  } else if constexpr (MM != NGT_MIP_NONE) {
    r = vzero<C>();
    // a position outside the finest level's valid range is outside every
    // level's, and most of a frustum is: no LoD, no reads (BORDER, LINEAR)
    if (!(FM == LINEAR && BM == BORDER) || xform_inside(a.din, px, py, pz)) {
      const float lod = xform_lod(a, cp, ix, iy, iz, px, py, pz);
      r = read_mip<C, FM, BM, MM>(mips, cp.data_index, px, py, pz, lod, a.mip_bias, 0.5f);
    }
  } else if constexpr (FM == LINEAR) {
    r = read_linear<C, BM>(a.input + cp.data_index * in_slice, a.din, px - 0.5f, py - 0.5f, pz - 0.5f);
  } else if constexpr (FM == QUADRATIC) {
    r = read_quadratic<C, BM>(a.input + cp.data_index * in_slice, a.din, px - 0.5f, py - 0.5f, pz - 0.5f);
  } else {
    r = read_nearest<C, BM>(a.input + cp.data_index * in_slice, a.din, px - 0.5f, py - 0.5f, pz - 0.5f);
  }
  const int64_t out_cells = static_cast<int64_t>(a.dout.x) * a.dout.y * a.dout.z;
  vstore<C>(out + (static_cast<int64_t>(cp.out_index) * out_cells + cell_offset(a.dout, x, y, z)) * C, r);
}

template <int C, int FM, int BM, bool REF, int MM>
__global__ __launch_bounds__(256) void xform_bwd_kernel(XformArgs a, CamBatch cb, MipSet grad,
                                                        const float* __restrict__ out_grad,
                                                        float* __restrict__ in_grad, uint32_t* __restrict__ hits) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  const int z = blockIdx.z % a.dout.z;
  const int ci = blockIdx.z / a.dout.z;
  if (x >= a.dout.x || y >= a.dout.y) return;
  const CamParams& cp = cb.cam[ci];
  const float ix = static_cast<float>(x) + 0.5f, iy = static_cast<float>(y) + 0.5f, iz = static_cast<float>(z) + 0.5f;
  float px, py, pz;
  xform_pos(a, cp, ix, iy, iz, px, py, pz);
  const int64_t in_cells = static_cast<int64_t>(a.din.x) * a.din.y * a.din.z;
  const int64_t out_cells = static_cast<int64_t>(a.dout.x) * a.dout.y * a.dout.z;
  const Vec<C> dy = vload<C>(out_grad + (static_cast<int64_t>(cp.out_index) * out_cells + cell_offset(a.dout, x, y, z)) * C);
  float* g = in_grad + cp.data_index * in_cells * C;
  if constexpr (REF) {
    // kScatter3DGradients: the quadratic scatter for QUADRATIC, the trilinear
    // one for every other filter (resample_grid.cu.cc:1160-1185)
    if constexpr (FM == QUADRATIC)
      scatter_quadratic_reference<C, BM>(g, a.din, px - 0.5f, py - 0.5f, pz - 0.5f, dy,
                                         hits + cp.data_index * in_cells);
    else
      scatter_linear<C, BM, true>(g, a.din, px - 0.5f, py - 0.5f, pz - 0.5f, dy, hits + cp.data_index * in_cells);
  } else if constexpr (BM != WRAP && MM != NGT_MIP_NONE) {
    const float lod = xform_lod(a, cp, ix, iy, iz, px, py, pz);
    const MipPick k = mip_pick<MM>(lod, a.mip_bias, grad.num_levels);
    // the transform filters need no level data for their scatter (LINEAR, NEAREST, QUADRATIC)
    scatter_level<C, FM, BM>(grad, grad, cp.data_index, k.lf, px, py, pz, 0.5f, vscale(dy, 1.f - k.wc));
    if (k.two) scatter_level<C, FM, BM>(grad, grad, cp.data_index, k.lc, px, py, pz, 0.5f, vscale(dy, k.wc));
  } else if constexpr (BM != WRAP) {
    if constexpr (FM == LINEAR) scatter_linear<C, BM, false>(g, a.din, px - 0.5f, py - 0.5f, pz - 0.5f, dy);
    else if constexpr (FM == QUADRATIC) scatter_quadratic<C, BM>(g, a.din, px - 0.5f, py - 0.5f, pz - 0.5f, dy);
    else scatter_nearest<C, BM>(g, a.din, px - 0.5f, py - 0.5f, pz - 0.5f, dy);
  }
}

// ------------------------------------------- transform adjoint as a gather ---
// The exact adjoint of LINEAR BORDER sampling in the forward modes, without
// global atomics: one work-group per brick of voxels of one level takes the
// output cells whose positions can fall into the brick's trilinear support -
// the bounding box, in output cells, of the support's 8 corners mapped through
// the camera - and adds the corner contributions of those that do to fp64
// accumulators in LDS (ds_add_f64, 3 to 7 lanes per clock and CU); the brick's
// voxels are then stored once, so nothing has to be cleared first.  Global
// fp32 atomics scatter at 21 to 85 G/s here: the frustum adjoint of a 96^3 grid
// of 4 channels with 2 mips into three 128x72x96 views took 1697 us, this 96:
// about 25 us of it finding the boxes and storing the voxels, 30 testing the
// candidates (2 to 3 for each sample in the support), the rest the LoDs, the
// gradients' loads and 11 us of LDS atomics.
//
// The accumulator is the brick grown by one cell on every side, so that the 8
// corners of every sample whose floor cell lies in b0 - 1 .. b1 land in it.
//
// A launch takes up to kMaxCamsPerLaunch (grid, camera) pairs and the bricks of
// the grids that these view, so that the bricks of all launches grow with the
// pairs: 64 grids of 64^3 into 32^3 cells around them, 4 channels, 223 us
// (with the bricks of every grid in each launch 64 grids of 64^3 into 16^3
// cells, 1 channel, took 648 us, without 137; these scatter now, in 55).
struct GridRange {
  int begin, count;  // the grids that the launch's pairs view
  int begin_new;     // the first of them that no earlier launch has stored
};

struct BrickList {
  int nx, ny, nz;
  __host__ __device__ int count() const { return nx * ny * nz; }
};

// The output index that object position p maps to, and the clip-space w (not
// positive behind the camera).  Linear depth is taken from view space, where
// it is affine in p.
template <typename T>
NGT_HOST_DEVICE_INLINE T output_index(const CamParams& cp, const Dims& d, bool linear_depth, T x, T y, T z, T o[3]) {
  T v[4], c[4];
  for (int r = 0; r < 4; ++r) v[r] = cp.mv[4 * r] * x + cp.mv[4 * r + 1] * y + cp.mv[4 * r + 2] * z + cp.mv[4 * r + 3];
  for (int r = 0; r < 4; ++r)
    c[r] = cp.p[4 * r] * v[0] + cp.p[4 * r + 1] * v[1] + cp.p[4 * r + 2] * v[2] + cp.p[4 * r + 3] * v[3];
  o[0] = (c[0] / c[3] * T(0.5) + T(0.5)) * d.x;
  o[1] = (c[1] / c[3] * T(0.5) + T(0.5)) * d.y;
  o[2] = linear_depth ? -(v[2] + cp.near_) / (cp.far_ - cp.near_) * d.z : (c[2] / c[3] * T(0.5) + T(0.5)) * d.z;
  return c[3];
}

// A brick of level m: BX x BY x BZ voxels of the finest level, 8x4x4 of the
// next and 4x4x4 of the ones after, whose voxels see 8 and 64 times the
// samples and which are few.
template <int BX, int BY, int BZ>
NGT_HOST_DEVICE_INLINE Dims level_brick(int m) {
  return m == 0 ? Dims{BX, BY, BZ} : (m == 1 ? Dims{8, 4, 4} : Dims{4, 4, 4});
}

template <int BX, int BY, int BZ>
NGT_HOST_DEVICE_INLINE BrickList level_bricks(const Dims& d, int m) {
  const Dims dm = level_dims(d, m), b = level_brick<BX, BY, BZ>(m);
  return BrickList{(dm.x + b.x - 1) / b.x, (dm.y + b.y - 1) / b.y, (dm.z + b.z - 1) / b.z};
}

// Work-groups that share the candidates of a brick of level m, which is split
// from level `first` on: its voxels have 8^m times the finest ones' candidates
// to try, and the coarse levels have few bricks.  Split levels are cleared
// first and take the shares' sums by atomics.  96^3 into three 128x72x96
// frustums, 1 channel, 3 / 4 / 6 levels: 228 / 274 / 306 us, unsplit 1582 / 6446
// / 11462 (the coarsest level's one brick tries every output cell).
NGT_HOST_DEVICE_INLINE int level_splits(int m, int first) {
  const int above = m - (first < 2 ? first : 2);
  return m < first ? 1 : (above < 2 ? 4 << (3 * above) : 256);
}

// Split from level 2 on where its bricks are few, or little of the time is the
// finer levels' (the same frustums with 2 levels, 1 channel: 183 us, split from
// level 3 on 274; 4 channels, 216 bricks, 304 against 276; 64^3 into 64^3 cells x
// 3, 4 channels, 64 bricks: 99 against 157), from level 1 on where its bricks
// leave half of the CUs idle (48^3 into 128x72x96 x 3, 1 channel, 1 / 2 / 3 levels:
// 146 / 200 / 250 us against 425 / 434 / 461; 24^3 into 24^3: 49 / 52 / 52 against
// 55 / 61 / 64), and from the finest on where that has few bricks and each of
// its voxels 4 or more cells of a view (16^3 into 64^3 x 3, 1 channel, 0 / 1 / 3
// levels: 52 / 90 / 100 us against 156 / 365 / 372; 16^3 that fill a 26^3-cell
// view, 4.3 cells a voxel, 0 / 1: 7.8 / 12.2 against 9.0 / 17.9, and 13.4 with the
// scatter).
inline int first_split_level(const Dims& d, const Dims& dout, int64_t n, int64_t c) {
  const auto bricks = [&](int m) { return level_bricks<8, 4, 4>(d, m).count() * n; };
  if (bricks(0) < 128 && dims_cells(dout) >= 4 * dims_cells(d)) return 0;
  return bricks(1) < 128 ? 1 : (c < 4 || bricks(2) < 128 ? 2 : 3);
}

// i / n and i % n for 0 <= i < 2^30, n > 0, from a float estimate that is off
// by at most a few hundred (by one for i below 2^22).
NGT_DEVICE int div_rem(int i, int n, float inv, int& rem) {
  int q = static_cast<int>(static_cast<float>(i) * inv);
  rem = i - q * n;
  while (rem < 0) { rem += n; --q; }
  while (rem >= n) { rem -= n; ++q; }
  return q;
}

template <int C, int MM, int BX, int BY, int BZ>
__global__ __launch_bounds__(256) void xform_bwd_gather_kernel(XformArgs a, CamBatch cb, MipSet grad,
                                                               const float* __restrict__ out_grad, GridRange grids,
                                                               int first_split) {
  static_assert(BX >= 8 && BY >= 4 && BZ >= 4, "the coarser levels' bricks fit the finest one's accumulator");
  // one plane per channel: consecutive cells on consecutive banks
  constexpr int NP = (BX + 2) * (BY + 2) * (BZ + 2);
  __shared__ double acc[NP * C];
  __shared__ int box[kMaxCamsPerLaunch][6];  // x0, y0, z0 and the extents (0: view skipped)
  const int tid = threadIdx.x;
  // the coarsest level's bricks, which see the most samples, come first
  int bid = blockIdx.x, m = grad.num_levels;
  BrickList bl = level_bricks<BX, BY, BZ>(grad.d0, m);
  while (m > 0 && bid >= bl.count() * level_splits(m, first_split) * grids.count) {
    bid -= bl.count() * level_splits(m, first_split) * grids.count;
    bl = level_bricks<BX, BY, BZ>(grad.d0, --m);
  }
  const int splits = level_splits(m, first_split), split = bid % splits;
  bid /= splits;
  const int n = grids.begin + bid / bl.count(), brem = bid % bl.count();
  const bool accumulate = n < grids.begin_new;
  Dims dm;
  float* const out = level_ptr<C>(grad, n, m, dm);
  const Dims lb = level_brick<BX, BY, BZ>(m);
  const int PX = lb.x + 2, PXY = PX * (lb.y + 2);
  const int b0x = brem % bl.nx * lb.x, b0y = brem / bl.nx % bl.ny * lb.y, b0z = brem / (bl.nx * bl.ny) * lb.z;
  const int b1x = min(b0x + lb.x, dm.x) - 1, b1y = min(b0y + lb.y, dm.y) - 1, b1z = min(b0z + lb.z, dm.z) - 1;
  for (int i = tid; i < NP * C; i += 256) acc[i] = 0.0;

  // lane = view * 8 + corner of the support box, in finest-level cells
  if (tid < 64) {
    const int ci = tid >> 3, c = tid & 7;
    const bool view = ci < cb.count && cb.cam[ci < cb.count ? ci : 0].data_index == n;
    const float s = static_cast<float>(1 << m);
    float lo[3] = {3.0e38f, 3.0e38f, 3.0e38f}, hi[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
    int unknown = 0;
    if (view) {
      const CamParams& cp = cb.cam[ci];
      const float px = s * ((c & 1) ? static_cast<float>(b1x) + 1.502f : static_cast<float>(b0x) - 0.502f);
      const float py = s * ((c & 2) ? static_cast<float>(b1y) + 1.502f : static_cast<float>(b0y) - 0.502f);
      const float pz = s * ((c & 4) ? static_cast<float>(b1z) + 1.502f : static_cast<float>(b0z) - 0.502f);
      float o[3];
      const float cw = output_index<float>(cp, a.dout, a.coord_mode != NGT_COORD_TRANSFORM, px, py, pz, o);
      // the grid stands before the camera (checked on the host), so only the
      // rounding of a corner next to the camera's plane gives a w that is not
      // positive or an index that is huge or no number: every cell is a candidate
      unknown = !(cw > 0.f) || !(fabsf(o[0]) < 1.0e9f) || !(fabsf(o[1]) < 1.0e9f) || !(fabsf(o[2]) < 1.0e9f);
#pragma unroll
      for (int k = 0; k < 3; ++k) lo[k] = hi[k] = o[k];
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        lo[k] = fminf(lo[k], __shfl_xor(lo[k], off, 64));
        hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], off, 64));
      }
      unknown |= __shfl_xor(unknown, off, 64);
    }
    if (c == 0 && ci < cb.count) {
      const int dims[3] = {a.dout.x, a.dout.y, a.dout.z};
      int ext[3], at[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        // cell i has its centre at index i + 0.5; 0.1 cells cover the rounding
        // of the two maps (checked on the host)
        const float f = static_cast<float>(dims[k]);
        const int i0 = unknown ? 0 : max(0, static_cast<int>(ceilf(fminf(fmaxf(lo[k], -2.f), f + 2.f) - 0.6f)));
        const int i1 = unknown ? dims[k] - 1
                               : min(dims[k] - 1, static_cast<int>(floorf(fminf(fmaxf(hi[k], -2.f), f + 2.f) - 0.4f)));
        at[k] = i0;
        ext[k] = view ? max(0, i1 - i0 + 1) : 0;
      }
      const bool empty = ext[0] == 0 || ext[1] == 0 || ext[2] == 0;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        box[ci][k] = at[k];
        box[ci][3 + k] = empty ? 0 : ext[k];
      }
    }
  }
  __syncthreads();

  const float sc = level_scale(m);
  const float fdx = static_cast<float>(dm.x), fdy = static_cast<float>(dm.y), fdz = static_cast<float>(dm.z);
  const int64_t out_cells = static_cast<int64_t>(a.dout.x) * a.dout.y * a.dout.z;
  bool any = false;
  for (int ci = 0; ci < cb.count; ++ci) {
    const int nx = box[ci][3], ny = box[ci][4], total = nx * ny * box[ci][5];
    if (total == 0) continue;
    any = true;
    const CamParams& cp = cb.cam[ci];
    const float* const g = out_grad + static_cast<int64_t>(cp.out_index) * out_cells * C;
    const float inv_nx = 1.f / static_cast<float>(nx), inv_ny = 1.f / static_cast<float>(ny);
    for (int i = split * 256 + tid; i < total; i += splits * 256) {
      int x, y;
      const int row = div_rem(i, nx, inv_nx, x);
      const int z = box[ci][2] + div_rem(row, ny, inv_ny, y);
      x += box[ci][0]; y += box[ci][1];
      // every candidate's gradient is loaded, so that the load is in flight
      // while the position is formed
      const Vec<C> dy = vload<C>(g + cell_offset(a.dout, x, y, z) * C);
      const float ix = static_cast<float>(x) + 0.5f, iy = static_cast<float>(y) + 0.5f, iz = static_cast<float>(z) + 0.5f;
      float px, py, pz;
      xform_pos(a, cp, ix, iy, iz, px, py, pz);
      const float qx = px * sc - 0.5f, qy = py * sc - 0.5f, qz = pz * sc - 0.5f;
      const float fx = floorf(qx), fy = floorf(qy), fz = floorf(qz);
      const float lx = fx - static_cast<float>(b0x - 1), ly = fy - static_cast<float>(b0y - 1),
                  lz = fz - static_cast<float>(b0z - 1);
      // the forward's validity, and the floor cell in b0 - 1 .. b1
      if (!((qx + 0.5f >= 0.f) & (qx + 0.5f < fdx) & (qy + 0.5f >= 0.f) & (qy + 0.5f < fdy) & (qz + 0.5f >= 0.f) &
            (qz + 0.5f < fdz) & (lx >= 0.f) & (lx <= static_cast<float>(b1x - b0x + 1)) & (ly >= 0.f) &
            (ly <= static_cast<float>(b1y - b0y + 1)) & (lz >= 0.f) & (lz <= static_cast<float>(b1z - b0z + 1))))
        continue;
      float weight = 1.f;
      if constexpr (MM != NGT_MIP_NONE) {
        const MipPick k = mip_pick<MM>(xform_lod(a, cp, ix, iy, iz, px, py, pz), a.mip_bias, grad.num_levels);
        if (k.lf == m) weight = 1.f - k.wc;
        else if (k.two && k.lc == m) weight = k.wc;
        else continue;
      }
      const Vec<C> val = vscale(dy, weight);
      const float wx = qx - fx, wy = qy - fy, wz = qz - fz;
      const float fw[2][3] = {{1.f - wx, 1.f - wy, 1.f - wz}, {wx, wy, wz}};
      // an integer coordinate's ceil corner is its floor corner
      const int sx = wx != 0.f ? 1 : 0, sy = wy != 0.f ? PX : 0, sz = wz != 0.f ? PXY : 0;
      double* const t = acc + static_cast<int>(lz) * PXY + static_cast<int>(ly) * PX + static_cast<int>(lx);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int bx = k & 1, by = (k >> 1) & 1, bz = k >> 2;
        const float w = fw[bx][0] * fw[by][1] * fw[bz][2];
        double* const q = t + (bx ? sx : 0) + (by ? sy : 0) + (bz ? sz : 0);
#pragma unroll
        for (int j = 0; j < C; ++j) lds_add(q + j * NP, val.v[j] * w);
      }
    }
  }
  if ((accumulate || splits > 1) && !any) return;  // uniform
  __syncthreads();
  for (int i = tid; i < lb.x * lb.y * lb.z; i += 256) {
    const int lx = i % lb.x, ly = i / lb.x % lb.y, lz = i / (lb.x * lb.y);  // powers of two, uniform
    const int x = b0x + lx, y = b0y + ly, z = b0z + lz;
    if (x > b1x || y > b1y || z > b1z) continue;
    const double* const t = acc + (lz + 1) * PXY + (ly + 1) * PX + lx + 1;
    float* const o = out + cell_offset(dm, x, y, z) * C;
    Vec<C> v;
#pragma unroll
    for (int j = 0; j < C; ++j) v.v[j] = static_cast<float>(t[j * NP]);
    if (splits > 1) {
#pragma unroll
      for (int j = 0; j < C; ++j)
        if (v.v[j] != 0.f) atomic_add(o + j, v.v[j]);
      continue;
    }
    if (accumulate) {
      const Vec<C> old = vload<C>(o);
#pragma unroll
      for (int j = 0; j < C; ++j) v.v[j] += old.v[j];
    }
    vstore<C>(o, v);
  }
}

// kComputeLoD3D (resample_grid.cu.cc:1706-1720): position and central
// difference LoD (calcLoD<CM>, sampling.hpp:72-139) per output cell.
__global__ __launch_bounds__(256) void lod_transform_kernel(XformArgs a, CamBatch cb, int relative,
                                                            float* __restrict__ out) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  const int z = blockIdx.z % a.dout.z;
  const int ci = blockIdx.z / a.dout.z;
  if (x >= a.dout.x || y >= a.dout.y) return;
  const CamParams& cp = cb.cam[ci];
  const float ix = static_cast<float>(x) + 0.5f, iy = static_cast<float>(y) + 0.5f, iz = static_cast<float>(z) + 0.5f;
  float d[3][3];
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    const float ex = e == 0 ? 1.f : 0.f, ey = e == 1 ? 1.f : 0.f, ez = e == 2 ? 1.f : 0.f;
    float mx, my, mz, qx, qy, qz;
    xform_pos(a, cp, ix - ex, iy - ey, iz - ez, mx, my, mz);
    xform_pos(a, cp, ix + ex, iy + ey, iz + ez, qx, qy, qz);
    d[e][0] = (mx - qx) * 0.5f; d[e][1] = (my - qy) * 0.5f; d[e][2] = (mz - qz) * 0.5f;
  }
  float l[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) l[k] = sqrtf(d[0][k] * d[0][k] + d[1][k] * d[1][k] + d[2][k] * d[2][k]);
  float px, py, pz;
  xform_pos(a, cp, ix, iy, iz, px, py, pz);
  if (relative) {
    px -= static_cast<float>(x); py -= static_cast<float>(y); pz -= static_cast<float>(z);
  }
  const int64_t out_cells = static_cast<int64_t>(a.dout.x) * a.dout.y * a.dout.z;
  *reinterpret_cast<float4*>(out + (static_cast<int64_t>(cp.out_index) * out_cells + cell_offset(a.dout, x, y, z)) * 4) =
      make_float4(px, py, pz, log2_lod(l[0], l[1], l[2]));
}

// ------------------------------------------------------------- dispatch -----

#define NGT_SWITCH_C(C_, ...)                                 \
  switch (C_) {                                               \
    case 1: { constexpr int CC = 1; __VA_ARGS__; } break;     \
    case 2: { constexpr int CC = 2; __VA_ARGS__; } break;     \
    default: { constexpr int CC = 4; __VA_ARGS__; } break;    \
  }
#define NGT_SWITCH_BM(B_, ...)                                      \
  switch (B_) {                                                     \
    case BORDER: { constexpr int BB = BORDER; __VA_ARGS__; } break; \
    case CLAMP: { constexpr int BB = CLAMP; __VA_ARGS__; } break;   \
    default: { constexpr int BB = WRAP; __VA_ARGS__; } break;       \
  }
#define NGT_SWITCH_FM(F_, ...)                                       \
  switch (F_) {                                                      \
    case LINEAR: { constexpr int FF = LINEAR; __VA_ARGS__; } break;  \
    case NEAREST: { constexpr int FF = NEAREST; __VA_ARGS__; } break; \
    case FMIN: { constexpr int FF = FMIN; __VA_ARGS__; } break;      \
    default: { constexpr int FF = FMAX; __VA_ARGS__; } break;        \
  }
#define NGT_SWITCH_FM3(F_, ...)                                      \
  switch (F_) {                                                      \
    case NEAREST: { constexpr int FF = NEAREST; __VA_ARGS__; } break; \
    case FMIN: { constexpr int FF = FMIN; __VA_ARGS__; } break;      \
    default: { constexpr int FF = FMAX; __VA_ARGS__; } break;        \
  }
#define NGT_SWITCH_FM2(F_, ...)                                      \
  switch (F_) {                                                      \
    case LINEAR: { constexpr int FF = LINEAR; __VA_ARGS__; } break;  \
    case QUADRATIC: { constexpr int FF = QUADRATIC; __VA_ARGS__; } break; \
    default: { constexpr int FF = NEAREST; __VA_ARGS__; } break;     \
  }
#define NGT_SWITCH_MM(M_, ...)                                                   \
  switch (M_) {                                                                  \
    case NGT_MIP_NONE: { constexpr int MMM = NGT_MIP_NONE; __VA_ARGS__; } break; \
    case NGT_MIP_NEAREST: { constexpr int MMM = NGT_MIP_NEAREST; __VA_ARGS__; } break; \
    default: { constexpr int MMM = NGT_MIP_LINEAR; __VA_ARGS__; } break;         \
  }
#define NGT_SWITCH_MM2(M_, ...)                                                          \
  switch (M_) {                                                                          \
    case NGT_MIP_NEAREST: { constexpr int MMM = NGT_MIP_NEAREST; __VA_ARGS__; } break; \
    default: { constexpr int MMM = NGT_MIP_LINEAR; __VA_ARGS__; } break;                 \
  }

int check_filter_boundary(int interpolation, int boundary) {
  NGT_REQUIRE(interpolation >= 0 && interpolation <= 3, NGT_ERR_INVALID_ARGUMENT, "invalid interpolation");
  NGT_REQUIRE(boundary >= 0 && boundary <= 2, NGT_ERR_INVALID_ARGUMENT, "invalid boundary");
  return NGT_OK;
}

// Mip arguments against an input shape (resample_grid.cc:338-347 plus the
// pyramid limits).
int check_mips(const int64_t* in_shape, int mipmapping, int num_mipmaps) {
  NGT_REQUIRE(mipmapping >= NGT_MIP_NONE && mipmapping <= NGT_MIP_LINEAR, NGT_ERR_INVALID_ARGUMENT,
              "invalid mipmapping");
  NGT_REQUIRE(mipmapping == NGT_MIP_NONE || num_mipmaps > 0, NGT_ERR_INVALID_ARGUMENT,
              "when using mipmaps num_mipmaps must be larger than 0.");
  if (mipmapping == NGT_MIP_NONE) return NGT_OK;
  NGT_REQUIRE(num_mipmaps <= kMaxMips, NGT_ERR_INVALID_ARGUMENT, "num_mipmaps must be at most 16");
  NGT_REQUIRE((in_shape[1] >> num_mipmaps) >= 1 && (in_shape[2] >> num_mipmaps) >= 1 &&
                  (in_shape[3] >> num_mipmaps) >= 1,
              NGT_ERR_INVALID_ARGUMENT,
              "num_mipmaps too large for the input grid (every mip level needs at least one cell per axis)");
  return NGT_OK;
}

int check_mip_grad(int mipmapping, int gradient_semantics) {
  NGT_REQUIRE(mipmapping == NGT_MIP_NONE || gradient_semantics != NGT_GRAD_REFERENCE, NGT_ERR_UNIMPLEMENTED,
              "the reference gradient supports mipmapping 'NONE' only (use exact gradient semantics for mips)");
  return NGT_OK;
}

size_t mip_bytes(const int64_t* in_shape, int mipmapping, int num_mipmaps) {
  if (in_shape == nullptr || mipmapping == NGT_MIP_NONE || num_mipmaps <= 0 || num_mipmaps > kMaxMips) return 0;
  const Shape5 si = shape5(in_shape);
  return align256(static_cast<size_t>(mip_floats(si.dims(), si.n, si.c, num_mipmaps)) * sizeof(float));
}

MipSet make_mips(const float* base, const int64_t* in_shape, void* levels, int num_mipmaps) {
  const Shape5 si = shape5(in_shape);
  return MipSet{const_cast<float*>(base), static_cast<float*>(levels), si.dims(), static_cast<int>(si.n),
                num_mipmaps};
}

int check_lut(const int64_t* in_shape, const int64_t* lut_shape, int mipmapping, int num_mipmaps,
              float cco, int separate, int normalized) {
  int rc = check_grid_shape(in_shape, "input");
  if (rc) return rc;
  NGT_REQUIRE(lut_shape && lut_shape[4] == 4 && lut_shape[0] > 0 && lut_shape[1] > 0 && lut_shape[2] > 0 &&
                  lut_shape[3] > 0,
              NGT_ERR_INVALID_ARGUMENT, "Invalid lut shape (NDHWC) with C=4");
  rc = check_mips(in_shape, mipmapping, num_mipmaps);
  if (rc) return rc;
  NGT_REQUIRE(!normalized || cco == 0.5f, NGT_ERR_INVALID_ARGUMENT,
              "Invalid cell center offset must be 0.5 when using normalized coordinates.");
  if (!separate)
    NGT_REQUIRE(lut_shape[0] == in_shape[0], NGT_ERR_INVALID_ARGUMENT,
                "camera batch must match data batch when not using global sampling.");
  return NGT_OK;
}

LutArgs make_lut_args(const float* input, const int64_t* in_shape, const float* lookup, const int64_t* lut_shape,
                      float cco, int separate, int relative, int normalized, float mip_bias) {
  LutArgs a;
  const Shape5 si = shape5(in_shape);
  a.input = input;
  a.din = si.dims();
  a.lut = lookup;
  a.dout = Dims{static_cast<int>(lut_shape[3]), static_cast<int>(lut_shape[2]), static_cast<int>(lut_shape[1])};
  a.n_data = static_cast<int>(si.n);
  a.n_cams = static_cast<int>(lut_shape[0]);
  a.separate = separate ? 1 : 0;
  a.cco = cco;
  a.relative = relative ? 1 : 0;
  a.normalized = normalized ? 1 : 0;
  a.mip_bias = mip_bias;
  return a;
}

int check_cams(const int64_t* in_shape, const float* M, const float* V, const float* P, const float* F,
               int num_cameras, const int32_t* out_dhw, int separate, std::vector<Pair>& pairs) {
  int rc = check_grid_shape(in_shape, "input");
  if (rc) return rc;
  NGT_REQUIRE(M && V && P && F, NGT_ERR_INVALID_ARGUMENT, "matrices and frustum must be given");
  NGT_REQUIRE(num_cameras > 0, NGT_ERR_INVALID_ARGUMENT, "camera batch size mismatch");
  NGT_REQUIRE(out_dhw && out_dhw[0] > 0 && out_dhw[1] > 0 && out_dhw[2] > 0, NGT_ERR_INVALID_ARGUMENT,
              "Invalid output_shape");
  return make_pairs(static_cast<int>(in_shape[0]), num_cameras, separate != 0, pairs);
}

int check_xform_attrs(int interpolation, int boundary, int coordinate_mode, float cell_center_offset,
                      const char* op) {
  NGT_REQUIRE(interpolation == LINEAR || interpolation == NEAREST || interpolation == QUADRATIC,
              NGT_ERR_INVALID_ARGUMENT, std::string(op) + " supports NEAREST, LINEAR and QUADRATIC interpolation");
  NGT_REQUIRE(boundary == BORDER || boundary == CLAMP, NGT_ERR_INVALID_ARGUMENT, "invalid boundary");
  NGT_REQUIRE(cell_center_offset == 0.5f, NGT_ERR_INVALID_ARGUMENT,
              "Invalid cell center offset for given coordinate mode.");
  NGT_REQUIRE(coordinate_mode == 0 || coordinate_mode == 1 || coordinate_mode == 3 || coordinate_mode == 4,
              NGT_ERR_INVALID_ARGUMENT, "Invalid coordinate_mode");
  return NGT_OK;
}

XformArgs make_xform_args(const float* input, const int64_t* in_shape, const int32_t* out_dhw, int coordinate_mode,
                          float mip_bias) {
  const Shape5 si = shape5(in_shape);
  XformArgs a;
  a.input = input;
  a.din = si.dims();
  a.dout = Dims{out_dhw[2], out_dhw[1], out_dhw[0]};
  a.out_inv_x = 1.f / a.dout.x; a.out_inv_y = 1.f / a.dout.y; a.out_inv_z = 1.f / a.dout.z;
  a.coord_mode = coordinate_mode;
  a.mip_bias = mip_bias;
  return a;
}

std::vector<CamParams> make_cams(const std::vector<Pair>& pairs, const float* M, const float* V, const float* P,
                                 const float* F) {
  std::vector<CamParams> cams;
  cams.reserve(pairs.size());
  for (const Pair& p : pairs) cams.push_back(make_cam(M + 16 * p.n, V + 16 * p.v, P + 16 * p.v, F + 6 * p.v, p.n, p.out));
  return cams;
}

CamBatch cam_batch(const std::vector<CamParams>& cams, size_t b) {
  CamBatch cb;
  cb.count = static_cast<int>(std::min<size_t>(kMaxCamsPerLaunch, cams.size() - b));
  for (int i = 0; i < cb.count; ++i) cb.cam[i] = cams[b + i];
  return cb;
}

// Whether output_index inverts the forward's positions (output cell -> grid
// through the inverse matrices, in float as the kernels form them) to 0.02
// cells on a 3x3x3 lattice of the output: the gather finds its candidates with
// the one, with 0.1 cells to spare, and takes them by the other.  (It does not
// for a singular matrix, whose inverse is taken as 0, nor where a depth range
// of many orders costs the projection its float digits.)
bool maps_agree(const CamParams& cp, const Dims& dout, int coord_mode) {
  const float dims[3] = {static_cast<float>(dout.x), static_cast<float>(dout.y), static_cast<float>(dout.z)};
  auto apply = [](const float* m, const float v[3], float o[4]) {
    for (int r = 0; r < 4; ++r) o[r] = m[4 * r] * v[0] + m[4 * r + 1] * v[1] + m[4 * r + 2] * v[2] + m[4 * r + 3];
  };
  const bool linear_depth = coord_mode != NGT_COORD_TRANSFORM;
  for (int i = 0; i < 27; ++i) {
    const int at[3] = {i % 3, i / 3 % 3, i / 9};
    float idx[3], ndc[3], v[4], o[4];
    for (int k = 0; k < 3; ++k) {
      idx[k] = 0.5f + std::floor(0.5f * static_cast<float>(at[k]) * (dims[k] - 1.f));
      ndc[k] = idx[k] / dims[k] * 2.f - 1.f;
    }
    if (linear_depth)
      ndc[2] = -cp.p[10] - cp.p[11] / -((cp.far_ - cp.near_) * (idx[2] / dims[2]) + cp.near_);
    apply(cp.p_inv, ndc, v);
    const float iw = 1.f / v[3];
    for (int k = 0; k < 3; ++k) v[k] *= iw;
    apply(cp.mv_inv, v, o);
    double back[3];
    const double w = output_index<double>(cp, dout, linear_depth, o[0], o[1], o[2], back);
    if (!(w > 0.0)) return false;
    for (int k = 0; k < 3; ++k)
      if (!(std::fabs(back[k] - idx[k]) < 0.02)) return false;
  }
  return true;
}

// Whether the sample support of every level's grid lies before the camera, so
// that each brick's projection is bounded by its corners'.
bool grid_in_front(const CamParams& cp, const Dims& din, const Dims& dout, int levels) {
  const double reach = 0.502 * static_cast<double>(int64_t(1) << levels);
  for (int c = 0; c < 8; ++c) {
    double o[3];
    if (!(output_index<double>(cp, dout, false, (c & 1) ? din.x + reach : -reach, (c & 2) ? din.y + reach : -reach,
                               (c & 4) ? din.z + reach : -reach, o) > 0.0))
      return false;
  }
  return true;
}

// Output cells in the box that a grid before the camera takes of its view: 1.4
// to 2.5 times the cells that sample it, and exactly these where the map is one
// of the axes.
double cells_around_grid(const CamParams& cp, const Dims& din, const Dims& dout, int coord_mode) {
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (int c = 0; c < 8; ++c) {
    double o[3];
    output_index<double>(cp, dout, coord_mode != NGT_COORD_TRANSFORM, (c & 1) ? din.x : 0, (c & 2) ? din.y : 0,
                         (c & 4) ? din.z : 0, o);
    for (int k = 0; k < 3; ++k) {
      lo[k] = std::min(lo[k], o[k]);
      hi[k] = std::max(hi[k], o[k]);
    }
  }
  const double dims[3] = {static_cast<double>(dout.x), static_cast<double>(dout.y), static_cast<double>(dout.z)};
  double cells = 1.0;
  for (int k = 0; k < 3; ++k) cells *= std::max(0.0, std::min(hi[k], dims[k]) - std::max(lo[k], 0.0));
  return cells;
}

// Whether output index and grid position differ by a scale and a shift per axis
// (resampling between grids): consecutive cells then scatter to consecutive
// voxels, which the atomics take several times faster.
bool maps_axes(const CamParams& cp) {
  for (int r = 0; r < 4; ++r)
    for (int c = 0; c < 4; ++c)
      if (r != c && (cp.p_inv[4 * r + c] != 0.f || (c < 3 && cp.mv_inv[4 * r + c] != 0.f))) return false;
  return true;
}

bool same_maps(const CamParams& a, const CamParams& b) {
  return std::memcmp(a.mv, b.mv, sizeof(a.mv)) == 0 && std::memcmp(a.mv_inv, b.mv_inv, sizeof(a.mv_inv)) == 0 &&
         std::memcmp(a.p, b.p, sizeof(a.p)) == 0 && std::memcmp(a.p_inv, b.p_inv, sizeof(a.p_inv)) == 0 &&
         std::memcmp(&a.near_, &b.near_, sizeof(a.near_)) == 0 && std::memcmp(&a.far_, &b.far_, sizeof(a.far_)) == 0;
}

// The gather serves LINEAR, BORDER and the forward modes, for cameras whose
// maps agree and that stand before the grid (a brick that the camera's plane
// cuts would try every output cell in one work-group), where the values that
// sample the grids are not too few: it visits every brick of every level, the
// scatter only the samples.  Other calls scatter.  The lines, in values (cells
// around the grid times channels) per voxel, and scatter / gather in us of
// 128^3 grids of one channel, the one grid in a 128^3-cell view scaled by t:
//   perspective, no mips   0.05   t = 0.4 (0.012): 11 / 17, 0.5 (0.025): 14 / 17, 0.75 (0.08): 27 / 17
//   perspective, 2 levels  0.15   0.5: 28 / 53, 0.75: 60 / 56, 1 (0.2): 93 / 64
//   axes, no mips          0.1    0.4 (0.06): 14 / 17, 0.5 (0.12): 18 / 17, 0.75 (0.42): 37 / 18
//   axes, 2 levels         1.5    0.5: 29 / 56, 1 (1): 75 / 118, 1.5 (3.4): 1372 / 294
// the last divided by the channels once more (four of them in 0.5: 143 / 69, the
// scatter's atomics then lying 16 bytes apart).  With more pairs than one launch
// takes, each launch also needs enough values to be worth its 6 us (12 with
// levels) against the scatter's 3: 128 grids of 32^3 with three views each of
// 16^3 / 32^3 / 48^3 cells, 48 launches, 1.48 / 1.15 / 0.27 times the scatter.
bool use_xform_gather(const std::vector<CamParams>& cams, const XformArgs& a, int64_t n_data, int channels, int levels,
                      int interpolation, int boundary) {
  if (interpolation != LINEAR || boundary != BORDER) return false;
  if (a.coord_mode != NGT_COORD_TRANSFORM && a.coord_mode != NGT_COORD_TRANSFORM_LINDEPTH) return false;
  if (dims_cells(a.dout) >= (int64_t(1) << 30) || dims_cells(a.din) * n_data >= (int64_t(1) << 36)) return false;
  // the views of the grids after the first are mostly the first one's again
  // (comparing takes 0.02 us of the host, checking 0.6)
  const size_t views = static_cast<size_t>(
      std::find_if(cams.begin(), cams.end(), [](const CamParams& c) { return c.data_index != 0; }) - cams.begin());
  const double voxels = static_cast<double>(dims_cells(a.din)) * static_cast<double>(n_data);
  double values = 0.0;
  bool axes = true;
  std::vector<double> cells(cams.size());
  for (size_t i = 0; i < cams.size(); ++i) {
    if (i >= views && same_maps(cams[i], cams[i - views])) {
      cells[i] = cells[i - views];
    } else {
      if (!maps_agree(cams[i], a.dout, a.coord_mode) || !grid_in_front(cams[i], a.din, a.dout, levels)) return false;
      cells[i] = cells_around_grid(cams[i], a.din, a.dout, a.coord_mode);
      axes = axes && maps_axes(cams[i]);
    }
    values += cells[i] * channels;
  }
  const double line = levels == 0 ? (axes ? 0.1 : 0.05) : (axes ? 1.5 / channels : 0.15);
  if (!(values >= line * voxels)) return false;
  const double launches = std::ceil(static_cast<double>(cams.size()) / kMaxCamsPerLaunch);
  return launches == 1.0 || values >= launches * (levels == 0 ? 32768.0 : 49152.0);
}

template <int C, int MM, int BX, int BY, int BZ>
void launch_xform_gather(const XformArgs& a, const CamBatch& cb, const MipSet& grad, const float* out_grad,
                         const GridRange& grids, int first_split, hipStream_t s) {
  int64_t bricks = 0;
  for (int m = 0; m <= grad.num_levels; ++m)
    bricks += static_cast<int64_t>(level_bricks<BX, BY, BZ>(grad.d0, m).count()) * level_splits(m, first_split) * grids.count;
  hipLaunchKernelGGL((xform_bwd_gather_kernel<C, MM, BX, BY, BZ>), dim3(static_cast<unsigned>(bricks)), dim3(256), 0, s,
                     a, cb, grad, out_grad, grids, first_split);
}

// The grids of the pairs from b on.  The pairs are in the order of their grids,
// so the launch before has stored at most the first of them.
GridRange grid_range(const std::vector<CamParams>& cams, size_t b) {
  const size_t e = std::min(cams.size(), b + kMaxCamsPerLaunch);
  const int begin = cams[b].data_index, end = cams[e - 1].data_index + 1;
  return GridRange{begin, end - begin, b > 0 ? cams[b - 1].data_index + 1 : 0};
}

}  // namespace
}  // namespace ngt

using namespace ngt;

extern "C" {

size_t ngt_sample_grid_lut_fwd_workspace_size(const int64_t* input_shape, int mipmapping, int num_mipmaps) {
  return mip_bytes(input_shape, mipmapping, num_mipmaps);
}

int ngt_sample_grid_lut_fwd(const float* input, const int64_t* input_shape, const float* lookup,
                            const int64_t* lookup_shape, int interpolation, int boundary, int mipmapping,
                            int num_mipmaps, float mip_bias, float cell_center_offset, int separate_camera_batch,
                            int relative_coords, int normalized_coords, float* output, void* workspace,
                            size_t workspace_bytes, ngt_stream_t stream) {
  int rc = check_lut(input_shape, lookup_shape, mipmapping, num_mipmaps, cell_center_offset, separate_camera_batch,
                     normalized_coords);
  if (rc) return rc;
  rc = check_filter_boundary(interpolation, boundary);
  if (rc) return rc;
  const size_t need = ngt_sample_grid_lut_fwd_workspace_size(input_shape, mipmapping, num_mipmaps);
  NGT_REQUIRE(workspace_bytes >= need && (need == 0 || workspace != nullptr), NGT_ERR_WORKSPACE,
              "workspace too small for ngt_sample_grid_lut_fwd");
  const LutArgs a = make_lut_args(input, input_shape, lookup, lookup_shape, cell_center_offset, separate_camera_batch,
                                  relative_coords, normalized_coords, mip_bias);
  const MipSet mips = make_mips(input, input_shape, workspace, mipmapping == NGT_MIP_NONE ? 0 : num_mipmaps);
  const int pairs = separate_camera_batch ? a.n_data * a.n_cams : a.n_data;
  const dim3 grid(blocks_for(a.dout.x, kBX), blocks_for(a.dout.y, kBY), static_cast<unsigned>(a.dout.z * pairs));
  const dim3 block(kBX, kBY);
  hipStream_t s = as_stream(stream);
  if (mipmapping != NGT_MIP_NONE) NGT_SWITCH_C(input_shape[4], launch_mip_generate<CC>(mips, s));
  NGT_SWITCH_C(input_shape[4], NGT_SWITCH_FM(interpolation, NGT_SWITCH_BM(boundary, NGT_SWITCH_MM(mipmapping,
      hipLaunchKernelGGL((lut_fwd_kernel<CC, FF, BB, MMM>), grid, block, 0, s, a, mips, output)))));
  return check_launch("ngt_sample_grid_lut_fwd");
}

size_t ngt_sample_grid_lut_bwd_workspace_size(const int64_t* input_shape, const int64_t* lookup_shape,
                                              int mipmapping, int num_mipmaps, int gradient_semantics) {
  (void)lookup_shape;
  if (input_shape == nullptr) return 0;
  if (gradient_semantics == NGT_GRAD_REFERENCE)
    return static_cast<size_t>(input_shape[0] * input_shape[1] * input_shape[2] * input_shape[3]) * sizeof(uint32_t);
  return 2 * mip_bytes(input_shape, mipmapping, num_mipmaps);  // level data + level gradients
}

int ngt_sample_grid_lut_bwd(const float* input, const int64_t* input_shape, const float* output_grad,
                            const float* lookup, const int64_t* lookup_shape, int interpolation, int boundary,
                            int mipmapping, int num_mipmaps, float mip_bias, float cell_center_offset,
                            int separate_camera_batch, int relative_coords, int normalized_coords,
                            int gradient_semantics, float* input_grad, float* lookup_grad, void* workspace,
                            size_t workspace_bytes, ngt_stream_t stream) {
  int rc = check_lut(input_shape, lookup_shape, mipmapping, num_mipmaps, cell_center_offset, separate_camera_batch,
                     normalized_coords);
  if (rc) return rc;
  rc = check_filter_boundary(interpolation, boundary);
  if (rc) return rc;
  rc = check_mip_grad(mipmapping, gradient_semantics);
  if (rc) return rc;
  const bool ref = gradient_semantics == NGT_GRAD_REFERENCE;
  const size_t need =
      ngt_sample_grid_lut_bwd_workspace_size(input_shape, lookup_shape, mipmapping, num_mipmaps, gradient_semantics);
  NGT_REQUIRE(workspace_bytes >= need && (need == 0 || workspace != nullptr), NGT_ERR_WORKSPACE,
              "workspace too small for ngt_sample_grid_lut_bwd");
  const LutArgs a = make_lut_args(input, input_shape, lookup, lookup_shape, cell_center_offset, separate_camera_batch,
                                  relative_coords, normalized_coords, mip_bias);
  const Shape5 si = shape5(input_shape);
  hipStream_t s = as_stream(stream);
  fill_zero(input_grad, si.elems(), s);
  const int slots = separate_camera_batch ? a.n_cams : a.n_data;
  const dim3 grid(blocks_for(a.dout.x, kBX), blocks_for(a.dout.y, kBY), static_cast<unsigned>(a.dout.z * slots));
  const dim3 block(kBX, kBY);
  if (mipmapping != NGT_MIP_NONE) {
    const size_t half = mip_bytes(input_shape, mipmapping, num_mipmaps);
    char* ws = static_cast<char*>(workspace);
    const MipSet data = make_mips(input, input_shape, ws, num_mipmaps);
    const MipSet grad = make_mips(input_grad, input_shape, ws + half, num_mipmaps);
    fill_zero(grad.levels, static_cast<int64_t>(mip_floats(si.dims(), si.n, si.c, num_mipmaps)), s);
    NGT_SWITCH_C(si.c, launch_mip_generate<CC>(data, s));
    if (interpolation == LINEAR) {
      NGT_SWITCH_C(si.c, NGT_SWITCH_BM(boundary, NGT_SWITCH_MM2(mipmapping,
          hipLaunchKernelGGL((lut_bwd_tile_kernel<CC, BB, MMM>), ScatterTile<CC>::grid(a.dout, slots), ScatterTile<CC>::block(),
                             0, s, a, data, grad, output_grad, lookup_grad))));
    } else {
      NGT_SWITCH_C(si.c, NGT_SWITCH_FM3(interpolation, NGT_SWITCH_BM(boundary, NGT_SWITCH_MM2(mipmapping,
          hipLaunchKernelGGL((lut_bwd_mip_kernel<CC, FF, BB, MMM>), grid, block, 0, s, a, data, grad, output_grad,
                             lookup_grad)))));
    }
    NGT_SWITCH_C(si.c, launch_mip_collapse<CC>(grad, s));
    return check_launch("ngt_sample_grid_lut_bwd");
  }
  uint32_t* hits = static_cast<uint32_t*>(workspace);
  if (ref) fill_zero_u32(hits, si.n * si.cells(), s);
  if (ref) {
    // the reference's input gradient is a trilinear scatter for every filter
    // mode; only LINEAR produces a LUT gradient
    if (interpolation == LINEAR) {
      NGT_SWITCH_C(si.c, NGT_SWITCH_BM(boundary,
          hipLaunchKernelGGL((lut_bwd_kernel<CC, LINEAR, BB, true>), grid, block, 0, s, a, output_grad, input_grad,
                             lookup_grad, hits)));
    } else {
      NGT_SWITCH_C(si.c, NGT_SWITCH_BM(boundary,
          hipLaunchKernelGGL((lut_bwd_kernel<CC, NEAREST, BB, true>), grid, block, 0, s, a, output_grad, input_grad,
                             lookup_grad, hits)));
    }
    NGT_SWITCH_C(si.c,
        hipLaunchKernelGGL((normalize_by_count_kernel<CC>), dim3(blocks_for(si.n * si.cells(), 256)), dim3(256), 0,
                           s, input_grad, hits, si.n * si.cells()));
  } else if (interpolation == LINEAR) {
    const MipSet data = make_mips(input, input_shape, nullptr, 0), grad = make_mips(input_grad, input_shape, nullptr, 0);
    NGT_SWITCH_C(si.c, NGT_SWITCH_BM(boundary,
        hipLaunchKernelGGL((lut_bwd_tile_kernel<CC, BB, NGT_MIP_NONE>), ScatterTile<CC>::grid(a.dout, slots), ScatterTile<CC>::block(), 0,
                           s, a, data, grad, output_grad, lookup_grad)));
  } else {
    NGT_SWITCH_C(si.c, NGT_SWITCH_FM3(interpolation, NGT_SWITCH_BM(boundary,
        hipLaunchKernelGGL((lut_bwd_kernel<CC, FF, BB, false>), grid, block, 0, s, a, output_grad, input_grad,
                           lookup_grad, nullptr))));
  }
  return check_launch("ngt_sample_grid_lut_bwd");
}

size_t ngt_sample_grid_transform_fwd_workspace_size(const int64_t* input_shape, int mipmapping, int num_mipmaps) {
  return mip_bytes(input_shape, mipmapping, num_mipmaps);
}

int ngt_sample_grid_transform_fwd(const float* input, const int64_t* input_shape, const float* matrix_m,
                                  const float* matrix_v, const float* matrix_p, const float* frustum,
                                  int num_cameras, const int32_t* output_dhw, int interpolation, int boundary,
                                  int mipmapping, int num_mipmaps, float mip_bias, int coordinate_mode,
                                  float cell_center_offset, int separate_camera_batch, float* output,
                                  void* workspace, size_t workspace_bytes, ngt_stream_t stream) {
  std::vector<Pair> pairs;
  int rc = check_cams(input_shape, matrix_m, matrix_v, matrix_p, frustum, num_cameras, output_dhw,
                      separate_camera_batch, pairs);
  if (rc) return rc;
  rc = check_xform_attrs(interpolation, boundary, coordinate_mode, cell_center_offset, "SampleGridTransform");
  if (rc) return rc;
  rc = check_mips(input_shape, mipmapping, num_mipmaps);
  if (rc) return rc;
  const size_t need = ngt_sample_grid_transform_fwd_workspace_size(input_shape, mipmapping, num_mipmaps);
  NGT_REQUIRE(workspace_bytes >= need && (need == 0 || workspace != nullptr), NGT_ERR_WORKSPACE,
              "workspace too small for ngt_sample_grid_transform_fwd");
  const Shape5 si = shape5(input_shape);
  const XformArgs a = make_xform_args(input, input_shape, output_dhw, coordinate_mode, mip_bias);
  const MipSet mips = make_mips(input, input_shape, workspace, mipmapping == NGT_MIP_NONE ? 0 : num_mipmaps);
  hipStream_t s = as_stream(stream);
  if (mipmapping != NGT_MIP_NONE) NGT_SWITCH_C(si.c, launch_mip_generate<CC>(mips, s));
  const std::vector<CamParams> cams = make_cams(pairs, matrix_m, matrix_v, matrix_p, frustum);
  for (size_t b = 0; b < cams.size(); b += kMaxCamsPerLaunch) {
    const CamBatch cb = cam_batch(cams, b);
    const dim3 grid(blocks_for(a.dout.x, kBX), blocks_for(a.dout.y, kBY), static_cast<unsigned>(a.dout.z * cb.count));
    const dim3 block(kBX, kBY);
    NGT_SWITCH_C(si.c, NGT_SWITCH_FM2(interpolation, NGT_SWITCH_BM(boundary, NGT_SWITCH_MM(mipmapping,
        hipLaunchKernelGGL((xform_fwd_kernel<CC, FF, BB, MMM>), grid, block, 0, s, a, cb, mips, output)))));
  }
  return check_launch("ngt_sample_grid_transform_fwd");
}

size_t ngt_sample_grid_transform_bwd_workspace_size(const int64_t* input_shape, int mipmapping, int num_mipmaps,
                                                    int gradient_semantics) {
  if (input_shape == nullptr) return 0;
  if (gradient_semantics == NGT_GRAD_REFERENCE)
    return static_cast<size_t>(input_shape[0] * input_shape[1] * input_shape[2] * input_shape[3]) * sizeof(uint32_t);
  return mip_bytes(input_shape, mipmapping, num_mipmaps);  // level gradients
}

int ngt_sample_grid_transform_bwd(const float* input, const int64_t* input_shape, const float* output_grad,
                                  const float* matrix_m, const float* matrix_v, const float* matrix_p,
                                  const float* frustum, int num_cameras, const int32_t* output_dhw,
                                  int interpolation, int boundary, int mipmapping, int num_mipmaps, float mip_bias,
                                  int coordinate_mode, float cell_center_offset, int separate_camera_batch,
                                  int gradient_semantics, float* input_grad, void* workspace, size_t workspace_bytes,
                                  ngt_stream_t stream) {
  std::vector<Pair> pairs;
  int rc = check_cams(input_shape, matrix_m, matrix_v, matrix_p, frustum, num_cameras, output_dhw,
                      separate_camera_batch, pairs);
  if (rc) return rc;
  rc = check_xform_attrs(interpolation, boundary, coordinate_mode, cell_center_offset, "SampleGridTransformGrad");
  if (rc) return rc;
  rc = check_mips(input_shape, mipmapping, num_mipmaps);
  if (rc) return rc;
  rc = check_mip_grad(mipmapping, gradient_semantics);
  if (rc) return rc;
  const bool ref = gradient_semantics == NGT_GRAD_REFERENCE;
  const size_t need =
      ngt_sample_grid_transform_bwd_workspace_size(input_shape, mipmapping, num_mipmaps, gradient_semantics);
  NGT_REQUIRE(workspace_bytes >= need && (need == 0 || workspace != nullptr), NGT_ERR_WORKSPACE,
              "workspace too small for ngt_sample_grid_transform_bwd");
  const Shape5 si = shape5(input_shape);
  const XformArgs a = make_xform_args(input, input_shape, output_dhw, coordinate_mode, mip_bias);
  const bool mip = mipmapping != NGT_MIP_NONE;
  const MipSet grad = make_mips(input_grad, input_shape, mip ? workspace : nullptr, mip ? num_mipmaps : 0);
  hipStream_t s = as_stream(stream);
  const std::vector<CamParams> cams = make_cams(pairs, matrix_m, matrix_v, matrix_p, frustum);
  if (!ref && use_xform_gather(cams, a, si.n, static_cast<int>(si.c), grad.num_levels, interpolation,
                               boundary)) {
    const int64_t at_once = grid_range(cams, 0).count;  // grids of a launch
    const int first_split = first_split_level(grad.d0, a.dout, at_once, si.c);
    const int64_t stored = mip_floats(si.dims(), si.n, si.c, std::max(first_split - 1, 0));
    const int64_t cleared = mip_floats(si.dims(), si.n, si.c, grad.num_levels) - stored;
    if (first_split == 0) fill_zero2(input_grad, si.elems(), grad.levels, cleared, s);
    else if (grad.num_levels >= first_split) fill_zero(grad.levels + stored, cleared, s);
    for (size_t b = 0; b < cams.size(); b += kMaxCamsPerLaunch) {
      const CamBatch cb = cam_batch(cams, b);
      // 8x8x8 bricks visit fewer samples twice and pay fewer prologues than
      // 8x4x4 ones (64^3 grid of 1 channel into 96^3 cells 17.5 us against
      // 21.2; 96^3 of 4 channels into frustums 96 against 110), which keep the
      // CUs busy on grids too small to give each two; 16x8x8 leave them too
      // few and too uneven (22.2 and 160 us)
      const bool large = level_bricks<8, 8, 8>(grad.d0, 0).count() * at_once >= 512;
      const GridRange grids = grid_range(cams, b);
      NGT_SWITCH_C(si.c, NGT_SWITCH_MM(mipmapping,
          if (large) launch_xform_gather<CC, MMM, 8, 8, 8>(a, cb, grad, output_grad, grids, first_split, s);
          else launch_xform_gather<CC, MMM, 8, 4, 4>(a, cb, grad, output_grad, grids, first_split, s)));
    }
    if (mip) NGT_SWITCH_C(si.c, launch_mip_collapse<CC>(grad, s));
    return check_launch("ngt_sample_grid_transform_bwd");
  }
  fill_zero(input_grad, si.elems(), s);
  uint32_t* hits = ref ? static_cast<uint32_t*>(workspace) : nullptr;
  if (ref) fill_zero_u32(hits, si.n * si.cells(), s);
  if (mip) fill_zero(grad.levels, static_cast<int64_t>(mip_floats(si.dims(), si.n, si.c, num_mipmaps)), s);
  for (size_t b = 0; b < cams.size(); b += kMaxCamsPerLaunch) {
    const CamBatch cb = cam_batch(cams, b);
    const dim3 grid(blocks_for(a.dout.x, kBX), blocks_for(a.dout.y, kBY), static_cast<unsigned>(a.dout.z * cb.count));
    const dim3 block(kBX, kBY);
    if (ref && interpolation == QUADRATIC) {
      NGT_SWITCH_C(si.c, NGT_SWITCH_BM(boundary,
          hipLaunchKernelGGL((xform_bwd_kernel<CC, QUADRATIC, BB, true, NGT_MIP_NONE>), grid, block, 0, s, a, cb,
                             grad, output_grad, input_grad, hits)));
    } else if (ref) {
      NGT_SWITCH_C(si.c, NGT_SWITCH_BM(boundary,
          hipLaunchKernelGGL((xform_bwd_kernel<CC, LINEAR, BB, true, NGT_MIP_NONE>), grid, block, 0, s, a, cb, grad,
                             output_grad, input_grad, hits)));
    } else {
      NGT_SWITCH_C(si.c, NGT_SWITCH_FM2(interpolation, NGT_SWITCH_BM(boundary, NGT_SWITCH_MM(mipmapping,
          hipLaunchKernelGGL((xform_bwd_kernel<CC, FF, BB, false, MMM>), grid, block, 0, s, a, cb, grad, output_grad,
                             input_grad, nullptr)))));
    }
  }
  if (mip) NGT_SWITCH_C(si.c, launch_mip_collapse<CC>(grad, s));
  if (ref) {
    NGT_SWITCH_C(si.c,
        hipLaunchKernelGGL((normalize_by_count_kernel<CC>), dim3(blocks_for(si.n * si.cells(), 256)), dim3(256), 0, s,
                           input_grad, hits, si.n * si.cells()));
  }
  return check_launch("ngt_sample_grid_transform_bwd");
}

int ngt_lod_transform(const int32_t* input_dhw, const float* matrix_mv, const float* matrix_p, const float* frustum,
                      int num_cameras, const int32_t* output_dhw, int inverse_transform, int linearize_depth,
                      int relative_coords, float* output, ngt_stream_t stream) {
  NGT_REQUIRE(input_dhw && input_dhw[0] > 0 && input_dhw[1] > 0 && input_dhw[2] > 0, NGT_ERR_INVALID_ARGUMENT,
              "Invalid input_shape");
  NGT_REQUIRE(output_dhw && output_dhw[0] > 0 && output_dhw[1] > 0 && output_dhw[2] > 0, NGT_ERR_INVALID_ARGUMENT,
              "Invalid output_shape");
  NGT_REQUIRE(matrix_mv && matrix_p && frustum, NGT_ERR_INVALID_ARGUMENT, "matrices and frustum must be given");
  NGT_REQUIRE(num_cameras > 0, NGT_ERR_INVALID_ARGUMENT, "camera batch size mismatch");
  const int cm = linearize_depth ? (inverse_transform ? NGT_COORD_TRANSFORM_LINDEPTH_REVERSE : NGT_COORD_TRANSFORM_LINDEPTH)
                                 : (inverse_transform ? NGT_COORD_TRANSFORM_REVERSE : NGT_COORD_TRANSFORM);
  const int64_t in_shape[5] = {1, input_dhw[0], input_dhw[1], input_dhw[2], 4};
  const XformArgs a = make_xform_args(nullptr, in_shape, output_dhw, cm, 0.f);
  static const float kIdentity[16] = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1};
  hipStream_t s = as_stream(stream);
  for (int b = 0; b < num_cameras; b += kMaxCamsPerLaunch) {
    CamBatch cb;
    cb.count = std::min(kMaxCamsPerLaunch, num_cameras - b);
    for (int i = 0; i < cb.count; ++i)
      cb.cam[i] = make_cam(kIdentity, matrix_mv + 16 * (b + i), matrix_p + 16 * (b + i), frustum + 6 * (b + i), 0,
                           b + i);
    const dim3 grid(blocks_for(a.dout.x, kBX), blocks_for(a.dout.y, kBY), static_cast<unsigned>(a.dout.z * cb.count));
    hipLaunchKernelGGL(lod_transform_kernel, grid, dim3(kBX, kBY), 0, s, a, cb, relative_coords ? 1 : 0, output);
  }
  return check_launch("ngt_lod_transform");
}

}  // extern "C"
