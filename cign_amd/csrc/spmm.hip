// CSR SpMM for the fixed graph operator: y = P x (+ add), and the chained
// three-hop pipeline built on it.
//
// Replaces the cuSPARSE SpMM calls of the reference MultiHopCsrPlan
// (multihop_csr_ext/multihop_csr_pipeline_cuda.cu:264-321) and the
// torch.sparse.mm recurrence of FixedCSRSpMMFunction (model.py:57-106).
//
// Layout: x, add, y are row-major [n_rows, ld] (fp32 or bf16 storage, fp32
// accumulation); P is CSR with int32 row pointer / column index and fp32
// values. One launch handles at most 256 16-byte chunks per row; wider
// matrices take several launches.
//
// A gather is bound by the cache lines it can have in flight, so by their
// latency: a launch of wide rows is split into column tiles that stay on
// their XCDs (workgroup ids go round-robin to the 8 XCDs), so that an XCD's
// 4 MB L2 holds more of the rows' slices it gathers (launch_all). 24,492
// nodes, 220,420 entries, fp32, us per hop forward / backward, untiled ->
// tiled: D = 512 56.1 / 61.9 -> 45.8 / 52.3 (8 tiles of 256 bytes), 384 40.5 /
// 44.0 -> 35.0 / 38.4, 256 26.6 / 28.7 -> 23.8 / 26.2; 2,000 nodes, D = 512:
// 14.4 -> 10.2 (too few wavefronts untiled); 60,000 nodes of 26 entries, D =
// 512: 394 / 407 -> 340 / 365.
//
// A row's output is owned by a group of L lanes (L = power of two covering
// the tile's chunks, 16-byte loads, lane l owns chunks l, l + L, ...). Three
// work shapes, from the degree-sorted schedule (schedule.h):
//   tiny rows   (degree <= L):  one row per lane group, G = 64 / L rows per
//                               wavefront; one col/val load, then the row's
//                               gathers in one batch;
//   medium rows (<= 64 edges):  one row per wavefront, its G groups split the
//                               edges, reduced with a butterfly;
//   heavy rows:                 segments (512 edges by the host default), one
//                               workgroup each, in rounds of 64 edges per
//                               wave; multi-segment rows merge through
//                               `partial` in segment order.
// A batch's gathers are unconditional (indices clamped to a valid edge,
// weight zero) so they all issue before the first is consumed; its size is
// the wavefront's largest per-group edge count rounded up to a power of two.
#include <mutex>

#include "common.h"
#include "schedule.h"

namespace cign {

// Values of rows that are not 16-byte aligned (odd widths, views): the same
// 16-byte accesses with the alignment of one value. Against one value a lane
// (24,492 nodes): fp32 D = 33 12.8 -> 7.9 us, 115 17.8 -> 13.7, 333 51.1 ->
// 37.5; bf16 D = 333 120 -> 29, 334 120 -> 25.
struct f32u {
  float v;
};
struct bf16u {
  uint16_t bits;
};
__device__ __forceinline__ float to_f32(f32u v) { return v.v; }
__device__ __forceinline__ float to_f32(bf16u v) { return __uint_as_float(static_cast<uint32_t>(v.bits) << 16); }
template <>
__device__ __forceinline__ f32u from_f32<f32u>(float f) { return f32u{f}; }
template <>
__device__ __forceinline__ bf16u from_f32<bf16u>(float f) { return bf16u{from_f32<bf16>(f).bits}; }

template <>
struct Chunk<f32u, 4> {
  using Raw = float4;
  typedef float Vec __attribute__((ext_vector_type(4), aligned(4)));
  static __device__ __forceinline__ Raw load_raw(const f32u* p) {
    const Vec q = *reinterpret_cast<const Vec*>(p);
    return make_float4(q.x, q.y, q.z, q.w);
  }
  static __device__ __forceinline__ Raw zero_raw() { return make_float4(0.0f, 0.0f, 0.0f, 0.0f); }
  static __device__ __forceinline__ void unpack(const Raw& q, float (&v)[4]) { Chunk<float, 4>::unpack(q, v); }
  static __device__ __forceinline__ void store(f32u* p, const float (&v)[4]) {
    *reinterpret_cast<Vec*>(p) = Vec{v[0], v[1], v[2], v[3]};
  }
};

template <>
struct Chunk<bf16u, 8> {
  using Raw = uint4;
  typedef uint32_t Vec __attribute__((ext_vector_type(4), aligned(2)));
  static __device__ __forceinline__ Raw load_raw(const bf16u* p) {
    const Vec q = *reinterpret_cast<const Vec*>(p);
    return make_uint4(q.x, q.y, q.z, q.w);
  }
  static __device__ __forceinline__ Raw zero_raw() { return make_uint4(0u, 0u, 0u, 0u); }
  static __device__ __forceinline__ void unpack(const Raw& q, float (&v)[8]) { Chunk<bf16, 8>::unpack(q, v); }
  static __device__ __forceinline__ void store(bf16u* p, const float (&v)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      w[i] = from_f32<bf16>(v[2 * i]).bits | (static_cast<uint32_t>(from_f32<bf16>(v[2 * i + 1]).bits) << 16);
    *reinterpret_cast<Vec*>(p) = Vec{w[0], w[1], w[2], w[3]};
  }
};

namespace {

// Workgroup shape of the SpMM: kSpmmWaves wavefronts; a heavy-row segment is
// processed in rounds of kSpmmWaves x 64 edges.
#ifndef CIGN_SPMM_WAVES
#define CIGN_SPMM_WAVES 8
#endif
constexpr int kSpmmWaves = CIGN_SPMM_WAVES;
// Chunks in flight per lane (a batch of U edges x VPL chunks).
#ifndef CIGN_SPMM_INFLIGHT
#define CIGN_SPMM_INFLIGHT 8
#endif
constexpr int kSpmmInflight = CIGN_SPMM_INFLIGHT;
constexpr int kSpmmBlock = kSpmmWaves * kWave;
constexpr int kTile = 64;
constexpr int kSegEdges = kSpmmWaves * kTile;

template <typename T, int W, int VPL, bool TILED>
struct SpmmArgs {
  int ld;       // row stride of x / add / y (elements)
  int c0;       // first column of the launch; in the kernel, of the workgroup's tile
  int nch;      // chunks (of W elements) of the launch; in the kernel, of the tile
  int lgT;      // log2 of the tiles, over which workgroup ids are dealt
  int width;    // columns of the launch (row stride of `partial`)
  int L;        // lanes per group (power of two, L * VPL >= nch)
  int lgL;      // log2(L)
  int n_mid;    // light rows processed one per wavefront (the first n_mid)
  int mid_blocks;
  const int32_t* col;
  const float* val;
  const T* x;
  const T* add;  // may be null
  T* y;
  float* partial;     // [n_seg, width] scratch for multi-segment rows
  int32_t* counters;  // [n_hrow], zero on entry, left zero on exit
};

template <int VPL, int W>
__device__ __forceinline__ void zero(float (&acc)[VPL][W]) {
#pragma unroll
  for (int v = 0; v < VPL; ++v)
#pragma unroll
    for (int w = 0; w < W; ++w) acc[v][w] = 0.0f;
}

// First column of the tile's chunk c within its row, from a.c0. Where the row
// is no whole number of chunks, the last chunk of the row ends at the row's
// end and repeats columns of the one before it, which is in the same launch
// (the same sums, in the same order, stored twice; both have loaded `add` by
// then).
template <typename T, int W, int VPL, bool TILED>
__device__ __forceinline__ int chunk_col(const SpmmArgs<T, W, VPL, TILED>& a, int c) {
  if constexpr (std::is_same<T, f32u>::value || std::is_same<T, bf16u>::value) return min(c * W, a.ld - W - a.c0);
  return c * W;
}

// Raw chunks of x[j] owned by lane gl (zero past the tile).
template <typename T, int W, int VPL, bool TILED>
__device__ __forceinline__ void load_row(const SpmmArgs<T, W, VPL, TILED>& a, int j, int gl,
                                         typename Chunk<T, W>::Raw (&buf)[VPL]) {
  const T* base = a.x + static_cast<int64_t>(j) * a.ld + a.c0;
#pragma unroll
  for (int v = 0; v < VPL; ++v) {
    const int c = gl + (v << a.lgL);
    buf[v] = c < a.nch ? Chunk<T, W>::load_raw(base + chunk_col(a, c)) : Chunk<T, W>::zero_raw();
  }
}

// Batches of U edge slots of a lane group: slot u = first + (k0 + k) * step,
// valid while u < cnt, whose column index and weight lane (base + u) holds in
// jj / vv. Every gather of a batch is issued before any is consumed; slots
// past the end reload an edge of the group with weight 0.
template <typename T, int W, int VPL, bool TILED>
struct SpmmBatches {
  const SpmmArgs<T, W, VPL, TILED>& a;
  int jj;
  float vv;
  int base, first, step, cnt, gl;
  float (&acc)[VPL][W];

  template <int U>
  __device__ __forceinline__ void run(int k0) {
    typename Chunk<T, W>::Raw buf[U][VPL];
    float wv[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const int u = first + (k0 + k) * step;
      const int src = (base + (u < cnt ? u : 0)) & (kWave - 1);
      const float v = shfl(vv, src);
      wv[k] = u < cnt ? v : 0.0f;
      load_row(a, shfl(jj, src), gl, buf[k]);
    }
#pragma unroll
    for (int k = 0; k < U; ++k)
#pragma unroll
      for (int v = 0; v < VPL; ++v) {
        float f[W];
        Chunk<T, W>::unpack(buf[k][v], f);
#pragma unroll
        for (int w = 0; w < W; ++w) acc[v][w] = fmaf(wv[k], f[w], acc[v][w]);
      }
  }
};

// Largest of v over the lane groups of a wavefront (runtime group size L).
__device__ __forceinline__ int wave_max_over_groups(int v, int L) {
  for (int o = L; o < kWave; o <<= 1) v = max(v, shfl_xor_i(v, o));
  return v;
}

// Gathers `need` (wave-uniform) slots per lane group, at most kSpmmInflight
// chunks in flight per lane.
template <typename T, int W, int VPL, bool TILED>
__device__ __forceinline__ void gather(const SpmmArgs<T, W, VPL, TILED>& a, int jj, float vv, int base, int first,
                                       int step, int cnt, int need, int gl, float (&acc)[VPL][W]) {
  SpmmBatches<T, W, VPL, TILED> sb{a, jj, vv, base, first, step, cnt, gl, acc};
  for_batches<(kSpmmInflight / VPL > 0 ? kSpmmInflight / VPL : 1)>(need, sb);
}

// The add row's chunks of a light row, loaded once the row is known and
// before its gathers (at the write they were one more memory round trip
// after the gathers, on every hop with a fused add). Chunks past the tile
// read the tile's last chunk (never used).
template <typename T, int W, int VPL, bool TILED>
struct AddRow {
  typename Chunk<T, W>::Raw raw[VPL];
  __device__ __forceinline__ void load(const SpmmArgs<T, W, VPL, TILED>& a, int row, int gl) {
    if (!a.add) return;  // uniform
    const T* base = a.add + static_cast<int64_t>(row) * a.ld + a.c0;
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
      const int c = min(gl + (v << a.lgL), a.nch - 1);
      raw[v] = Chunk<T, W>::load_raw(base + chunk_col(a, c));
    }
  }
};

template <typename T, int W, int VPL, bool TILED>
__device__ __forceinline__ void write_row(const SpmmArgs<T, W, VPL, TILED>& a, int row, int gl,
                                          const float (&acc)[VPL][W], const AddRow<T, W, VPL, TILED>& ar) {
#pragma unroll
  for (int v = 0; v < VPL; ++v) {
    const int c = gl + (v << a.lgL);
    if (c < a.nch) {
      const int64_t off = static_cast<int64_t>(row) * a.ld + a.c0 + chunk_col(a, c);
      float out[W];
#pragma unroll
      for (int w = 0; w < W; ++w) out[w] = acc[v][w];
      if (a.add) {
        float ad[W];
        Chunk<T, W>::unpack(ar.raw[v], ad);
#pragma unroll
        for (int w = 0; w < W; ++w) out[w] += ad[w];
      }
      Chunk<T, W>::store(a.y + off, out);
    }
  }
}

template <typename T, int W, int VPL, bool TILED>
__global__ __launch_bounds__(kSpmmBlock) void spmm_kernel(SpmmArgs<T, W, VPL, TILED> a, Sched s) {
  const int lane = lane_id();
  const int wave = wave_id();
  const int gl = lane & (a.L - 1);
  const int G = kWave >> a.lgL;
  const int g = lane >> a.lgL;
  // Workgroup ids go round-robin to the XCDs, so a tile stays on the same
  // XCDs (launch_all).
  int b = blockIdx.x;
  const int launch_c0 = a.c0;
  if constexpr (TILED) {
    const int tile = b & ((1 << a.lgT) - 1);
    b >>= a.lgT;
    a.nch >>= a.lgT;
    a.c0 += tile * a.nch * W;
  }
  float acc[VPL][W];
  zero(acc);

  if (b >= s.n_seg) {
    b -= s.n_seg;
    if (b < a.mid_blocks) {
      // Medium row (L < degree <= 64): one per wavefront, group g takes edges
      // g, g + G, ...
      const int li = b * kSpmmWaves + wave;
      if (li >= a.n_mid) return;
      const int4 r = s.light[li];
      const int deg = r.z - r.y;
      const bool mine = lane < deg;
      const int jj = mine ? a.col[r.y + lane] : 0;
      const float vv = mine ? a.val[r.y + lane] : 0.0f;
      AddRow<T, W, VPL, TILED> ar;
      ar.load(a, r.x, gl);
      gather(a, jj, vv, 0, g, G, deg, (deg + G - 1) / G, gl, acc);
      sum_across_n(acc, a.L);
      if (lane < a.L) write_row(a, r.x, gl, acc, ar);
      return;
    }
    // Tiny rows (degree <= L; in tiled launches every light row): one per lane
    // group.
    const int li = a.n_mid + ((b - a.mid_blocks) * kSpmmWaves + wave) * G + g;
    const bool has = li < s.n_light;
    const int4 r = has ? s.light[li] : make_int4(0, 0, 0, 0);
    const int deg = r.z - r.y;
    const bool mine = gl < deg;
    int jj = mine ? a.col[r.y + gl] : 0;
    float vv = mine ? a.val[r.y + gl] : 0.0f;
    AddRow<T, W, VPL, TILED> ar;
    ar.load(a, r.x, gl);  // (row 0 for a group with no row: read, unused)
    if constexpr (TILED) {
      // Every light row, L edges a round (the next round's indices loaded
      // ahead); the wavefront's rows have about the same degree. A row's terms
      // are then added in edge order, as in a launch of one tile.
      const int top = wave_max_over_groups(deg, a.L);
      for (int k = 0; k < top; k += a.L) {
        const int kn = k + a.L + gl;
        const int jn = kn < deg ? a.col[r.y + kn] : jj;
        const float vn = kn < deg ? a.val[r.y + kn] : 0.0f;
        gather(a, jj, vv, g << a.lgL, 0, 1, max(0, min(deg - k, a.L)), min(top - k, a.L), gl, acc);
        jj = jn;
        vv = vn;
      }
    } else {
      gather(a, jj, vv, g << a.lgL, 0, 1, deg, wave_max_over_groups(deg, a.L), gl, acc);
    }
    // A group's slots past its row's end reload an edge of that row; a row with
    // no edge has read another row's. (Rows of several chunks a lane have whole
    // wavefronts, so no light row comes here but in tiled launches; the sums'
    // second life costs bf16 rows 2 registers and with them a sixth wavefront per
    // SIMD: D = 640 39.0 us without, 42.8 with.)
    if constexpr (TILED || VPL == 1) {
      if (deg == 0) zero(acc);
    }
    if (has) write_row(a, r.x, gl, acc, ar);
    return;
  }

  // Heavy-row segment: wave w takes the segment's edges [64w, 64w + 64) of
  // every round of kSegEdges, reduced through LDS.
  __shared__ float red[kSpmmWaves][VPL * W * kWave];
  __shared__ int flag;
  const int4 sg = s.seg[b];
  const int row = sg.x;
  // Several rounds where the schedule's segments are longer than one.
  // The next round's indices and weights are loaded before this round's
  // gathers, so a round waits on one memory latency instead of two.
  int tb = sg.y + wave * kTile;
  int jj = tb + lane < sg.z ? a.col[tb + lane] : 0;
  float vv = tb + lane < sg.z ? a.val[tb + lane] : 0.0f;
  for (; tb < sg.z; tb += kSegEdges) {
    const int cnt = min(kTile, sg.z - tb);
    const int tn = tb + kSegEdges + lane;
    const int jn = tn < sg.z ? a.col[tn] : 0;
    const float vn = tn < sg.z ? a.val[tn] : 0.0f;
    gather(a, jj, vv, 0, g, G, cnt, (cnt + G - 1) / G, gl, acc);
    jj = jn;
    vv = vn;
  }
  sum_across_n(acc, a.L);
  // Columns of the tile; column c is value red_at(c) of its chunks.
  const int width = min(a.nch * W, a.ld - a.c0);
  const int full = (a.nch - 1) * W;
  const int skip = a.nch * W - width;
  const auto red_at = [&](int c) { return c < full ? c : c + skip; };
  if (lane < a.L) {
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
      const int c = lane + (v << a.lgL);
      if (c < a.nch)
#pragma unroll
        for (int w = 0; w < W; ++w) red[wave][c * W + w] = acc[v][w];
    }
  }
  __syncthreads();
  const int2 hr = s.hrow[sg.w];
  if (hr.y == 1) {
    for (int c = threadIdx.x; c < width; c += kSpmmBlock) {
      float t = 0.0f;
#pragma unroll
      for (int v = 0; v < kSpmmWaves; ++v) t += red[v][red_at(c)];
      const int64_t off = static_cast<int64_t>(row) * a.ld + a.c0 + c;
      if (a.add) t += to_f32(a.add[off]);
      a.y[off] = from_f32<T>(t);
    }
    return;
  }
  // The last of the row's workgroups, over all of its tiles, adds the
  // partials of the whole row (one counter per row).
  float* part = a.partial + static_cast<int64_t>(b) * a.width + (a.c0 - launch_c0);
  for (int c = threadIdx.x; c < width; c += kSpmmBlock) {
    float t = 0.0f;
#pragma unroll
    for (int v = 0; v < kSpmmWaves; ++v) t += red[v][red_at(c)];
    st_agent(part + c, t);
  }
  if (!arrive_last(a.counters + sg.w, hr.y << a.lgT, &flag)) return;
  for (int c = threadIdx.x; c < a.width; c += kSpmmBlock) {
    float t = 0.0f;
    for (int q = 0; q < hr.y; ++q) t += ld_agent(a.partial + static_cast<int64_t>(hr.x + q) * a.width + c);
    const int64_t off = static_cast<int64_t>(row) * a.ld + launch_c0 + c;
    if (a.add) t += to_f32(a.add[off]);
    a.y[off] = from_f32<T>(t);
  }
}

inline int ilog2(int v) {
  int r = 0;
  while ((1 << r) < v) ++r;
  return r;
}

struct SchedInfo {
  const int32_t* hdr;
  int n_light, n_seg, n_hrow;
};

inline SchedInfo read_info(const int32_t* hdr) { return SchedInfo{hdr, hdr[0], hdr[1], hdr[2]}; }

template <typename T, int W, int VPL, bool TILED>
int launch_tiles(hipStream_t stream, const Sched& s, const SchedInfo& info, int ld, int c0, int nch, int lgT,
                 const int32_t* col, const float* val, const T* x, const T* add, T* y, float* partial,
                 int32_t* counters) {
  SpmmArgs<T, W, VPL, TILED> a;
  a.ld = ld;
  a.c0 = c0;
  a.nch = nch;
  a.lgT = lgT;
  a.width = min(nch * W, ld - c0);
  const int lanes_needed = ((nch >> lgT) + VPL - 1) / VPL;
  // Unaligned rows of three or four chunks (bf16) take a group of eight lanes:
  // in a smaller one no light row shares its wavefront (n_mid below).
  constexpr int kMinLgL = std::is_same<T, f32u>::value || std::is_same<T, bf16u>::value ? 3 : 0;
  a.lgL = max(kMinLgL, ilog2(lanes_needed < 1 ? 1 : lanes_needed));
  a.L = 1 << a.lgL;
  a.col = col;
  a.val = val;
  a.x = x;
  a.add = add;
  a.y = y;
  a.partial = partial;
  a.counters = counters;
  const int G = kWave / a.L;
  // Rows with degree <= L go one per lane group (tiny); the rest of the
  // light list (sorted by degree, descending) one per wavefront.
  const int n_mid = TILED ? 0 : (G > 1 && a.L >= 8) ? sched_count_gt(info.hdr, a.L) : info.n_light;
  a.n_mid = n_mid;
  a.mid_blocks = (n_mid + kSpmmWaves - 1) / kSpmmWaves;
  const int n_tiny = info.n_light - n_mid;
  const int tiny_blocks = (n_tiny + kSpmmWaves * G - 1) / (kSpmmWaves * G);
  const int64_t blocks = static_cast<int64_t>(s.n_seg + a.mid_blocks + tiny_blocks) << lgT;
  if (blocks == 0) return kOk;
  if (blocks > INT32_MAX) return set_error(kInvalid, "cign_spmm: %lld workgroups", static_cast<long long>(blocks));
  hipLaunchKernelGGL((spmm_kernel<T, W, VPL, TILED>), dim3(static_cast<unsigned>(blocks)), dim3(kSpmmBlock), 0, stream,
                     a, s);
  return check_launch("cign_spmm");
}

template <typename T, int W>
int launch_all(hipStream_t stream, const Sched& s, const SchedInfo& info, int ld, const int32_t* col,
               const float* val, const T* x, const T* add, T* y, float* partial, int32_t* counters) {
  const int total_ch = (ld + W - 1) / W;
  constexpr int kMaxCh = kWave * 4;  // chunks per launch
  constexpr int kChunkBytes = static_cast<int>(sizeof(T)) * W;
  constexpr bool kTiles = W > 1 && std::is_same<T, float>::value;
  constexpr int kTileBytes = 256;
  constexpr int kLineCh = 128 / kChunkBytes;  // chunks of a 128-byte line (tiled launches)
  for (int ch0 = 0, nch; ch0 < total_ch; ch0 += nch) {
    nch = min(kMaxCh, total_ch - ch0);
    // A last chunk that overlaps the one before it (chunk_col) shares its
    // launch: in a launch of its own it would add `add` again to columns that
    // are stored, where y is add.
    if (ld % W != 0 && total_ch - ch0 - nch == 1) --nch;
    const int c0 = ch0 * W;
    // Column tiles of one launch: up to 8, none narrower than 256 bytes (two
    // tiles of 128 at D = 64: 10.9 us against 8.8), and each a whole number of
    // 128-byte lines, aligned to them: tiles that share lines fetch those from
    // two XCDs (D = 200: 22.8 us whole, 24.0 in two tiles; at 24,492 nodes and
    // 100,000 of 17 entries D = 160 19.9 and 136 us whole, 21.0 and 152 in two
    // tiles of 320 bytes; 288 31.4 and 247 whole, 34.2 and 297 in four; 640 61.4
    // and 534 in four, 66.4 and 616 in eight). Rows of at most 512 bytes stay
    // whole (D = 128: 13.5 us either way), and so do bf16 rows, whose lanes
    // unpack twice the values of a load (24,492 nodes, D = 512: 29.4 us whole or
    // in two tiles, 46.8 in eight).
    int lgT = 0;
    if constexpr (kTiles) {
      if (nch * kChunkBytes > 512 && (ld * static_cast<int>(sizeof(T))) % 128 == 0)
        while (lgT < 3 && (nch >> (lgT + 1)) * kChunkBytes >= kTileBytes && (nch >> lgT) % (2 * kLineCh) == 0) ++lgT;
    }
    const int tch = nch >> lgT;
    const int vpl = tch <= (lgT == 0 ? kWave : 16) ? 1 : tch <= 2 * kWave ? 2 : 4;
    int rc = kOk;
#define CIGN_SPMM_LAUNCH(VPL, TILED)                                                                             \
  rc = launch_tiles<T, W, VPL, TILED>(stream, s, info, ld, c0, nch, lgT, col, val, x, add, y, partial, counters)
    if (lgT == 0) {
      if (vpl == 1) CIGN_SPMM_LAUNCH(1, false);
      else if (vpl == 2) CIGN_SPMM_LAUNCH(2, false);
      else CIGN_SPMM_LAUNCH(4, false);
    } else if constexpr (kTiles) {
      if (vpl == 1) CIGN_SPMM_LAUNCH(1, true);
      else CIGN_SPMM_LAUNCH(2, true);
    }
#undef CIGN_SPMM_LAUNCH
    if (rc != kOk) return rc;
  }
  return kOk;
}

template <typename T>
int spmm_dispatch(hipStream_t stream, const Sched& s, const SchedInfo& info, int d, const int32_t* col,
                  const float* val, const void* x, const void* add, void* y, float* partial, int32_t* counters) {
  constexpr int kVec = 16 / sizeof(T);
  const T* xt = static_cast<const T*>(x);
  const T* at = static_cast<const T*>(add);
  T* yt = static_cast<T*>(y);
  const bool aligned = (reinterpret_cast<uintptr_t>(x) % 16 == 0) && (reinterpret_cast<uintptr_t>(y) % 16 == 0) &&
                       (add == nullptr || reinterpret_cast<uintptr_t>(add) % 16 == 0);
  if (d % kVec == 0 && aligned) {
    return launch_all<T, kVec>(stream, s, info, d, col, val, xt, at, yt, partial, counters);
  }
  // One value a lane up to 16 columns: a lane group of those widths has eight or
  // sixteen lanes either way, and chunks leave most of them idle (one value a
  // lane / chunks, us at 24,492 and 100,000 nodes: fp32 D = 5 6.3 and 30 / 9.6
  // and 39, 15 7.0 and 32 / 9.4 and 44, 17 8.9 and 45 / 7.2 and 41).
  if (d > 16) {
    using U = typename std::conditional<sizeof(T) == 4, f32u, bf16u>::type;
    return launch_all<U, kVec>(stream, s, info, d, col, val, reinterpret_cast<const U*>(xt),
                               reinterpret_cast<const U*>(at), reinterpret_cast<U*>(yt), partial, counters);
  }
  return launch_all<T, 1>(stream, s, info, d, col, val, xt, at, yt, partial, counters);
}

__global__ __launch_bounds__(kBlock) void zero_i32_kernel(int32_t* p, int n) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = 0;
}

}  // namespace
}  // namespace cign

// Scratch of cign_spmm_fwd3_noalloc: kNoAllocCounterInts int32 merge
// counters, then the segment partial sums of multi-segment rows. Each GPU
// the library runs on holds its own copy until the process ends. In host
// code `scratch` names a host-side stand-in, never the device memory: host
// code uses only the address hipGetSymbolAddress returns for the current
// device (noalloc_scratch below).
constexpr int64_t kNoAllocScratchBytes = 16ll << 20;
constexpr int64_t kNoAllocCounterInts = 1ll << 18;
constexpr int64_t kNoAllocPartialBytes = kNoAllocScratchBytes - kNoAllocCounterInts * 4;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace cign {
namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device, looked up once per device
// and kept for the life of the process: a hipDeviceReset (or unloading the
// library's code object) invalidates it, and the entry point must not be
// called on that device afterwards.
int noalloc_scratch(const char* what, void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return set_error(kHipError, "%s: hipGetDevice: %s", what, hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return set_error(kInvalid, "%s: device ordinal %d out of range", what, dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      return set_error(kHipError, "%s: hipGetSymbolAddress(scratch) on device %d: %s", what, dev,
                       hipGetErrorString(e));
    }
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return kOk;
}

}  // namespace
}  // namespace cign

using namespace cign;

extern "C" {

// Bytes of fp32 scratch `partial` needed by cign_spmm for a schedule with
// n_seg segments and d dense columns.
int64_t cign_spmm_partial_bytes(int32_t n_seg, int32_t d) {
  const int64_t tile = static_cast<int64_t>(d < kWave * 4 * 8 ? d : kWave * 4 * 8);
  return static_cast<int64_t>(n_seg) * tile * 4;
}

// y = P x (+ add). Replaces one cusparseSpMM of MultiHopCsrPlan::spmm
// (multihop_csr_ext/multihop_csr_pipeline_cuda.cu:264-285) or one
// torch.sparse.mm (model.py:91,101).
int cign_spmm(void* stream, int32_t dtype, int32_t n_rows, int32_t d, const int32_t* col, const float* val,
              const int32_t* sched, const int32_t* sched_info, const void* x, const void* add, void* y,
              float* partial, int32_t* counters) {
  if (n_rows < 0 || d <= 0) return set_error(kInvalid, "cign_spmm: bad sizes n_rows=%d d=%d", n_rows, d);
  if (!sched_info) return set_error(kInvalid, "cign_spmm: null schedule header");
  const SchedInfo info = read_info(sched_info);
  if (info.n_light + info.n_hrow != n_rows)
    return set_error(kInvalid, "cign_spmm: schedule does not cover %d rows", n_rows);
  if (!sched || !x || !y) return set_error(kInvalid, "cign_spmm: null pointer");
  if (info.n_seg > 0 && (!partial || !counters))
    return set_error(kInvalid, "cign_spmm: heavy rows need partial/counters");
  const Sched s = make_sched(sched, info.n_light, info.n_seg, info.n_hrow);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == kF32) return spmm_dispatch<float>(st, s, info, d, col, val, x, add, y, partial, counters);
  if (dtype == kBF16) return spmm_dispatch<bf16>(st, s, info, d, col, val, x, add, y, partial, counters);
  return set_error(kInvalid, "cign_spmm: unsupported dtype %d", dtype);
}

// Three chained hops without host work: y1 = P x, y2 = P y1, y3 = P y2.
// Replaces MultiHopCsrPlan::forward3 (multihop_csr_pipeline_cuda.cu:287-297).
int cign_spmm_fwd3(void* stream, int32_t dtype, int32_t n_rows, int32_t d, const int32_t* col, const float* val,
                   const int32_t* sched, const int32_t* sched_info, const void* x, void* y1, void* y2, void* y3,
                   float* partial, int32_t* counters) {
  int rc = cign_spmm(stream, dtype, n_rows, d, col, val, sched, sched_info, x, nullptr, y1, partial, counters);
  if (rc) return rc;
  rc = cign_spmm(stream, dtype, n_rows, d, col, val, sched, sched_info, y1, nullptr, y2, partial, counters);
  if (rc) return rc;
  return cign_spmm(stream, dtype, n_rows, d, col, val, sched, sched_info, y2, nullptr, y3, partial, counters);
}

// Chain-rule backward on P^T with the "+ g_k" adds fused into the SpMM
// epilogue: t2 = g2 + P^T g3, t1 = g1 + P^T t2, gx = P^T t1.
// Replaces MultiHopCsrPlan::backward3 (multihop_csr_pipeline_cuda.cu:299-321).
int cign_spmm_bwd3(void* stream, int32_t dtype, int32_t n_rows, int32_t d, const int32_t* col, const float* val,
                   const int32_t* sched, const int32_t* sched_info, const void* g1, const void* g2, const void* g3,
                   void* t2, void* t1, void* gx, float* partial, int32_t* counters) {
  int rc = cign_spmm(stream, dtype, n_rows, d, col, val, sched, sched_info, g3, g2, t2, partial, counters);
  if (rc) return rc;
  rc = cign_spmm(stream, dtype, n_rows, d, col, val, sched, sched_info, t2, g1, t1, partial, counters);
  if (rc) return rc;
  return cign_spmm(stream, dtype, n_rows, d, col, val, sched, sched_info, t1, nullptr, gx, partial, counters);
}

// cign_spmm_fwd3 with its partial sums and merge counters in the library's
// own per-GPU scratch, so the call allocates nothing. The counters are
// cleared by a fill kernel on `stream` first. Calls that overlap on one GPU
// (different streams or threads) share the scratch and race.
int cign_spmm_fwd3_noalloc(void* stream, int32_t dtype, int32_t n_rows, int32_t d, const int32_t* col,
                           const float* val, const int32_t* sched, const int32_t* sched_info, const void* x,
                           void* y1, void* y2, void* y3) {
  static const char* kWhat = "cign_spmm_fwd3_noalloc";
  if (!sched_info) return set_error(kInvalid, "%s: null schedule header", kWhat);
  if (d <= 0) return set_error(kInvalid, "%s: bad dense width d=%d", kWhat, d);
  const SchedInfo info = read_info(sched_info);
  if (info.n_seg < 0 || info.n_hrow < 0) return set_error(kInvalid, "%s: corrupt schedule header", kWhat);
  const int64_t counter_ints = static_cast<int64_t>(info.n_hrow) + 1;
  const int64_t partial_bytes = cign_spmm_partial_bytes(info.n_seg, d);
  if (counter_ints > kNoAllocCounterInts || partial_bytes > kNoAllocPartialBytes) {
    return set_error(kInvalid,
                     "%s: this schedule needs %lld merge counters and %lld bytes of partial sums; the built-in "
                     "scratch holds %lld counters and %lld bytes (use cign_spmm_fwd3 with caller workspace)",
                     kWhat, static_cast<long long>(counter_ints), static_cast<long long>(partial_bytes),
                     static_cast<long long>(kNoAllocCounterInts), static_cast<long long>(kNoAllocPartialBytes));
  }
  void* base = nullptr;
  int rc = noalloc_scratch(kWhat, &base);
  if (rc) return rc;
  int32_t* counters = static_cast<int32_t*>(base);
  float* partial = reinterpret_cast<float*>(static_cast<unsigned char*>(base) + kNoAllocCounterInts * 4);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int nc = static_cast<int>(counter_ints);
  hipLaunchKernelGGL(zero_i32_kernel, dim3((nc + kBlock - 1) / kBlock), dim3(kBlock), 0, st, counters, nc);
  rc = check_launch(kWhat);
  if (rc) return rc;
  return cign_spmm_fwd3(stream, dtype, n_rows, d, col, val, sched, sched_info, x, y1, y2, y3, partial, counters);
}

}  // extern "C"
