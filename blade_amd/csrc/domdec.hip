// domdec.hip - cell sort, blocks, tile list and exclusion masks
// (restates domdec/assign_domain.cu:14-45, assign_blocks.cu:24-468,
// cull.cu:44-375, assign_excl.cu:17-371, recull.cu:41-146 on 32-bit
// fractional coordinates; orc_domdec in the oracle is the same rule set).
//
// Rebuild sequence (no host synchronisation, fixed grids, graph-capturable):
//   dd_wrap_count -> [dd_scan_columns] -> dd_scatter -> dd_sort_columns ->
//   dd_tile_count -> dd_tile_write
// Few dependent launches: each one costs about 5 us beside its own work
// (start-up, drain, a dependent load chain), which is most of a rebuild at
// the usual sizes, so prefix sums over columns (up to kScanCols) and rows
// are formed by every workgroup that needs them (a few KB from L2) instead
// of in kernels of their own, and the exclusion masks are made by the wave
// that writes the row.
// Every step: dd_pack (slot positions, block boxes, accumulator reset).
//
// The tile list is directed: row I holds every block J (J == I included)
// whose rebuild box is within rcut + pad, in ascending J, so each pair of
// blocks appears as (I,J) and (J,I).  Rows are cut into chunks of at most
// d.tchunk tiles; the nonbonded kernel owns one chunk (one i-block) at a
// time and never writes j-side forces.
//
// Column counts and bucket fills walk the slots of the previous rebuild,
// which are ordered by column, so the lanes of a wave mostly share one
// column and one atomic serves them all (device-scope atomics on one
// address serialise across the chip).
#include "kernels.h"

#pragma clang fp contract(off)

namespace blade {

// Sums of N values over the 256 threads of a workgroup, for all of them
// (every thread must call it; s_sum: 4 N ints of LDS, free again on return).
template <int N>
__device__ __forceinline__ void wg_sum256(int (&v)[N], int *s_sum) {
#pragma unroll
  for (int k = 0; k < N; k++) {
    for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o, 64);
    if ((threadIdx.x & 63) == 0) s_sum[(threadIdx.x >> 6) * N + k] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; k++) v[k] = s_sum[k] + s_sum[N + k] + s_sum[2 * N + k] + s_sum[3 * N + k];
  __syncthreads();
}

// Exclusive prefix sum of f(0..n) into out[0..n], out[n] the total, by the
// 256 threads of a workgroup; out may be in LDS or global memory.
template <class F>
__device__ __forceinline__ void wg_scan256(int n, F f, int *out, int *s_sum) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int run = 0;
  for (int i0 = 0; i0 < n; i0 += 256) {
    const int i = i0 + threadIdx.x;
    const int v = i < n ? f(i) : 0;
    int x = v;
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) s_sum[w] = x;
    __syncthreads();
    int pre = run;
    for (int k = 0; k < 4; k++) {
      if (k < w) pre += s_sum[k];
      run += s_sum[k];
    }
    if (i < n) out[i] = pre + x - v;
    __syncthreads();
  }
  if (threadIdx.x == 0) out[n] = run;
}

// wrap every atom into the box, fractional coordinates, column counts and
// each atom's place in its column's bucket (one thread per slot of the
// previous rebuild; every atom has one slot; the pack clears the counts)
__device__ __forceinline__ void dd_wrap_count_body(const Dev &d, int bid, int nblk) {
  if (halted_wg(d)) return;   // a halted step leaves the list as it is
  const int s = bid * blockDim.x + threadIdx.x;
  const int i = s < 32 * d.maxblocks ? d.l2g[s] : -1;
  int col = 0;
  if (i >= 0) {
    unsigned u[3];
    for (int k = 0; k < 3; k++) {
      double x = d.pos[k * d.n + i];
      nan_check(d, x, i);
      double w = floor(__dmul_rn(x, d.invbox[k]));
      x = __dsub_rn(x, __dmul_rn(w, d.box[k]));
      d.pos[k * d.n + i] = x;
      u[k] = frac_u32(x, d.invbox[k]);
      d.ufrac[k * d.n + i] = u[k];
    }
    unsigned cx = (unsigned)(((unsigned long long)u[0] * (unsigned)d.ncx) >> 32);
    unsigned cy = (unsigned)(((unsigned long long)u[1] * (unsigned)d.ncy) >> 32);
    col = cx * d.ncy + cy;
  }
  const int f = wave_claim(d.colcount, col, i >= 0);
  if (i >= 0) d.colrank[i] = f;
}
__global__ void __launch_bounds__(256) dd_wrap_count(Dev d) { dd_wrap_count_body(d, blockIdx.x, gridDim.x); }
__global__ void __launch_bounds__(256) dd_wrap_count_multi(Multi m) {
  const MultiBlk b = multi_block(m);
  const Dev d = m.devs[b.sys];
  dd_wrap_count_body(d, b.bid, b.nblk);
}

// Column starts and, with ceil(count/32) blocks to a column, block starts;
// start: [ncol+1] in LDS or global memory, all 256 threads.
__device__ __forceinline__ void dd_column_starts(const Dev &d, int *start, int *s_sum) {
  wg_scan256(d.ncol, [&](int c) { return d.colcount[c]; }, start, s_sum);
  __syncthreads();
}
__device__ __forceinline__ void dd_block_starts(const Dev &d, int *s_sum) {
  wg_scan256(d.ncol, [&](int c) { return (d.colcount[c] + kBlockAtoms - 1) / kBlockAtoms; }, d.blkstart, s_sum);
  if (threadIdx.x == 0) *d.nblocks = d.blkstart[d.ncol];   // this thread's own store
}

// Most columns whose counts every workgroup of dd_scatter scans for itself
// (16 KB of LDS); of more, a kernel of one workgroup stores the starts first.
// A rebuild with and without that kernel: 49.3 and 47.8 us at 961 columns,
// 104.1 and 102.2 at 3,025, 243 and 242 at 5,625.
constexpr int kScanCols = 4096;

__device__ __forceinline__ void dd_scan_columns_body(const Dev &d) {
  if (halted_wg(d)) return;   // a halted step leaves the list as it is
  __shared__ int s_sum[4];
  dd_column_starts(d, d.colstart, s_sum);
  dd_block_starts(d, s_sum);
}
__global__ void __launch_bounds__(256) dd_scan_columns(Dev d) { dd_scan_columns_body(d); }
__global__ void __launch_bounds__(256) dd_scan_columns_multi(Multi m) {
  const MultiBlk b = multi_block(m);
  const Dev d = m.devs[b.sys];
  dd_scan_columns_body(d);
}

// Atoms into column buckets (bucket order is arbitrary; the column sort
// fixes the final order).  Up to kScanCols columns, every workgroup scans
// their counts into LDS, and the first also stores the starts.
__device__ __forceinline__ void dd_scatter_body(const Dev &d, int bid) {
  if (halted_wg(d)) return;   // a halted step leaves the list as it is
  __shared__ int s_start[kScanCols + 1], s_sum[4];
  const bool own = d.ncol <= kScanCols;
  if (own) dd_column_starts(d, s_start, s_sum);
  const int s = bid * blockDim.x + threadIdx.x;
  const int i = s < 32 * d.maxblocks ? d.l2g[s] : -1;
  if (i >= 0) {
    const unsigned cx = (unsigned)(((unsigned long long)d.ufrac[i] * (unsigned)d.ncx) >> 32);
    const unsigned cy = (unsigned)(((unsigned long long)d.ufrac[d.n + i] * (unsigned)d.ncy) >> 32);
    const int c = cx * d.ncy + cy;
    d.bucket[(own ? s_start[c] : d.colstart[c]) + d.colrank[i]] = i;
  }
  if (own && bid == 0) {
    for (int c = threadIdx.x; c <= d.ncol; c += blockDim.x) d.colstart[c] = s_start[c];
    dd_block_starts(d, s_sum);
  }
}
__global__ void __launch_bounds__(256) dd_scatter(Dev d) { dd_scatter_body(d, blockIdx.x); }
__global__ void __launch_bounds__(256) dd_scatter_multi(Multi m) {
  const MultiBlk b = multi_block(m);
  const Dev d = m.devs[b.sys];
  dd_scatter_body(d, b.bid);
}

// One workgroup per column: rank atoms by (z fraction, atom index), place
// them into 32-slot blocks, then the exact rebuild box of every block from
// the fractions held in LDS (one half-wave per block).
__device__ __forceinline__ void dd_sort_columns_body(const Dev &d, int bid, int nblk) {
  if (halted_wg(d)) return;   // a halted step leaves the list as it is
  __shared__ unsigned long long key[kMaxColumnAtoms];
  __shared__ unsigned sx[kMaxColumnAtoms], sy[kMaxColumnAtoms];
  __shared__ short sorted[kMaxColumnAtoms];
  const int c = bid;
  const int start = d.colstart[c], cnt = d.colcount[c];
  const int b0 = d.blkstart[c], nbc = d.blkstart[c + 1] - b0;
  if (cnt > kMaxColumnAtoms) {
    if (threadIdx.x == 0) atomicOr(d.errflag, 1);
    return;
  }
  for (int k = threadIdx.x; k < cnt; k += blockDim.x) {
    int a = d.bucket[start + k];
    key[k] = ((unsigned long long)d.ufrac[2 * d.n + a] << 32) | (unsigned)a;
    sx[k] = d.ufrac[a];
    sy[k] = d.ufrac[d.n + a];
  }
  __syncthreads();
  for (int k = threadIdx.x; k < cnt; k += blockDim.x) {
    unsigned long long kk = key[k];
    int rank = 0;
    for (int m = 0; m < cnt; m++) rank += key[m] < kk;
    int a = (int)(kk & 0xFFFFFFFFull);
    int slot = (b0 + rank / kBlockAtoms) * kBlockAtoms + rank % kBlockAtoms;
    d.l2g[slot] = a;
    d.g2s[a] = slot;
    sorted[rank] = (short)k;
  }
  for (int s = threadIdx.x; s < nbc * kBlockAtoms; s += blockDim.x)
    if (s >= cnt) d.l2g[b0 * kBlockAtoms + s] = -1;
  // slots past the last block may hold atoms of an earlier, longer list:
  // the next rebuild walks every slot, so clear them
  if (c == 0)
    for (int s = *d.nblocks * kBlockAtoms + threadIdx.x; s < d.maxblocks * kBlockAtoms; s += blockDim.x)
      d.l2g[s] = -1;
  __syncthreads();
  // block boxes: half-wave h of the workgroup takes blocks h, h+8, ...
  const int h = threadIdx.x >> 5, l = threadIdx.x & 31;
  for (int bb = h; bb < ((nbc + 7) / 8) * 8; bb += 8) {
    const int r = bb * kBlockAtoms + l;
    const bool in = bb < nbc && r < cnt;
    unsigned lo[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}, hi[3] = {0u, 0u, 0u};
    if (in) {
      const int k = sorted[r];
      const unsigned u[3] = {sx[k], sy[k], (unsigned)(key[k] >> 32)};
      for (int q = 0; q < 3; q++) lo[q] = hi[q] = u[q];
    }
    for (int q = 0; q < 3; q++)
      for (int o = 16; o > 0; o >>= 1) {
        lo[q] = min(lo[q], (unsigned)__shfl_xor((int)lo[q], o, 32));
        hi[q] = max(hi[q], (unsigned)__shfl_xor((int)hi[q], o, 32));
      }
    // clusters of eight for the pair kernel: the block's atoms in two halves
    // by x, each half in two by y (a block is a z slice of its column, so
    // the clusters are prisms half as wide as the column); empty slots last
    if (d.clusters) {
      const unsigned kx = in ? sx[sorted[r]] : 0xFFFFFFFFu, ky = in ? sy[sorted[r]] : 0xFFFFFFFFu;
      int rx = 0;
      for (int o = 0; o < kBlockAtoms; o++) {
        const unsigned v = (unsigned)__shfl((int)kx, o, 32);
        rx += v < kx || (v == kx && o < l);
      }
      int ry = 0;
      for (int o = 0; o < kBlockAtoms; o++) {
        const unsigned v = (unsigned)__shfl((int)ky, o, 32);
        const int ox = __shfl(rx, o, 32);
        ry += (ox >> 4) == (rx >> 4) && (v < ky || (v == ky && o < l));
      }
      if (bb < nbc) d.sperm[(b0 + bb) * kBlockAtoms + (rx & 16) + ry] = (unsigned char)l;
    }
    if (bb < nbc && l < 3) {
      d.bblo[3 * (b0 + bb) + l] = l == 0 ? lo[0] : l == 1 ? lo[1] : lo[2];
      d.bbhi[3 * (b0 + bb) + l] = l == 0 ? hi[0] : l == 1 ? hi[1] : hi[2];
    }
  }
}
__global__ void __launch_bounds__(256) dd_sort_columns(Dev d) { dd_sort_columns_body(d, blockIdx.x, gridDim.x); }
__global__ void __launch_bounds__(256) dd_sort_columns_multi(Multi m) {
  const MultiBlk b = multi_block(m);
  const Dev d = m.devs[b.sys];
  dd_sort_columns_body(d, b.bid, b.nblk);
}

// Periodic gap between two rebuild boxes (fractional counts), squared, in
// A^2, against (rcut+pad)^2; rounding as in the oracle (no contraction).
// The gap to either side is a difference modulo 2^32.  Pairs clearly inside
// or outside in FP32 (whose error is below 1e-6 relative) are settled
// there; the rest in the oracle's FP64 arithmetic.
// core: the boxes are within rcut as they stand.
__device__ __forceinline__ bool dd_close(const Dev &d, const unsigned (&aLo)[3], const unsigned (&aHi)[3],
                                         const unsigned (&bLo)[3], const unsigned (&bHi)[3], bool &core) {
  unsigned gap[3];
  float sf = 0.f;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const bool apart = aHi[k] < bLo[k] || bHi[k] < aLo[k];
    gap[k] = apart ? min(bLo[k] - aHi[k], aLo[k] - bHi[k]) : 0u;
    const float g = (float)gap[k] * d.fracscale[k];
    sf += g * g;
  }
  const float r2 = (float)d.rlist2;
  core = sf <= d.rc2;
  if (sf < r2 * 0.99999f) return true;
  if (sf > r2 * 1.00001f) return false;
  double g[3];
#pragma unroll
  for (int k = 0; k < 3; k++) g[k] = __dmul_rn((double)gap[k], d.ddscale[k]);
  double s = __dadd_rn(__dmul_rn(g[0], g[0]), __dmul_rn(g[1], g[1]));
  s = __dadd_rn(s, __dmul_rn(g[2], g[2]));
  return s <= d.rlist2;
}

__device__ __forceinline__ void dd_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The tile kernels take the blocks J of a row in windows, whose boxes and
// bitmaps they hold in LDS, so that neither grows with the system.  1,024
// blocks (about 30,000 atoms of water to a window) take 27 KB for the counts
// and 35 KB for the writer with its masks: five and four workgroups to a CU.
// Counts and writer at 3,100 rows: 34 and 45 us, with windows of 2,048 blocks
// 31 and 60 (two workgroups of the writer to a CU), with every row's bitmap
// and 3,072 boxes in LDS 57 and 94 (one).  At 740 rows and fewer, one window
// either way: 12 and 20 us.
constexpr int kWindow = 1024;
constexpr int kRowChunks = 64;   // chunks of a row counted one by one (later ones share the last count)
constexpr int kRows = 4;         // rows (waves) of a workgroup

// block boxes [W0, W0 + kWindow) into LDS (every thread of the block must
// call it); 16 bytes a load, four in flight: word by word this was most of
// the tile kernels' time at 2,900 blocks
__device__ __forceinline__ void dd_stage_boxes(const Dev &d, int W0, int nb, unsigned *lo, unsigned *hi) {
  if (W0) __syncthreads();   // the window before has been used
  const int m = 3 * min(nb - W0, kWindow), m4 = m / 4;
  const uint4 *glo = reinterpret_cast<const uint4 *>(d.bblo + 3 * (size_t)W0);
  const uint4 *ghi = reinterpret_cast<const uint4 *>(d.bbhi + 3 * (size_t)W0);
#pragma unroll 4
  for (int k = threadIdx.x; k < m4; k += 256) {
    reinterpret_cast<uint4 *>(lo)[k] = glo[k];
    reinterpret_cast<uint4 *>(hi)[k] = ghi[k];
  }
  if ((int)threadIdx.x < m - 4 * m4) {
    const size_t k = 4 * m4 + threadIdx.x;
    lo[k] = d.bblo[3 * (size_t)W0 + k];
    hi[k] = d.bbhi[3 * (size_t)W0 + k];
  }
  __syncthreads();
}

// LDS of one row's window: the bitmap of its blocks J (64-bit words), the
// tiles before each word, a bit per tile for exclusions; and the tiles within
// rcut of each chunk of the row
struct DdRowLds {
  unsigned long long bits[kRows][kWindow / 64], ebits[kRows][kWindow / 64];
  int pre[kRows][kWindow / 64], core[kRows][kRowChunks];
};

struct DdRow {
  unsigned long long *bits, *ebits;   // kept blocks; tiles with exclusions, by place in the window
  int *pre, *core;                    // tiles of the window before a word of bits; tiles of a chunk within rcut
  int W0, base, cnt;                  // the window; tiles of the row before it; tiles in it

  __device__ __forceinline__ DdRow(DdRowLds &l, int w)
      : bits(l.bits[w]), ebits(l.ebits[w]), pre(l.pre[w]), core(l.core[w]), W0(0), base(0), cnt(0) {
    core[threadIdx.x & 63] = 0;
  }
  // place in the window of the tile to block J, -1 if it has none
  __device__ __forceinline__ int place(int J) const {
    const unsigned j = J - W0;
    if (j >= (unsigned)kWindow) return -1;
    const unsigned long long m = bits[j >> 6], bit = 1ull << (j & 63);
    return m & bit ? pre[j >> 6] + __popcll(m & (bit - 1)) : -1;
  }
  // chunk k has more than half its tiles within rcut
  __device__ __forceinline__ bool is_long(const Dev &d, int k) const {
    return 2 * core[min(k, kRowChunks - 1)] > d.tchunk;
  }
};
static_assert(kRowChunks == 64, "a lane clears each chunk's count");

// Exclusions of slot lane % 32 of a block, two lanes to a slot on alternate
// ones, eight loads in flight each (an atom of a chain has a dozen or more,
// each behind two dependent loads): f(partner's slot).
template <class F>
__device__ __forceinline__ void dd_exclusions(const Dev &d, int I, F f) {
  constexpr int kBatch = 8;
  const int lane = threadIdx.x & 63, a = d.l2g[I * kBlockAtoms + (lane & (kBlockAtoms - 1))];
  const int x0 = a >= 0 ? d.exstart[a] + (lane >> 5) : 0, x1 = a >= 0 ? d.exstart[a + 1] : 0;
  for (int x = x0; x < x1; x += 2 * kBatch) {
    int sb[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; k++) sb[k] = x + 2 * k < x1 ? d.exadj[x + 2 * k] : a;
#pragma unroll
    for (int k = 0; k < kBatch; k++) sb[k] = d.g2s[sb[k]];
#pragma unroll
    for (int k = 0; k < kBatch; k++)
      if (x + 2 * k < x1) f(sb[k]);
  }
}

// One wave, row I, window W0: the blocks J of the window within the list
// radius in ascending order (tile(place in the row, J) for each), their
// chunks' tiles within rcut, and the tiles holding an excluded pair.
template <class F>
__device__ __forceinline__ void dd_scan_row(const Dev &d, const unsigned *lo, const unsigned *hi, int W0, int nb, int I,
                                            DdRow &r, F tile) {
  const int lane = threadIdx.x & 63;
  unsigned aLo[3], aHi[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    aLo[k] = d.bblo[3 * I + k];
    aHi[k] = d.bbhi[3 * I + k];
  }
  r.base += r.cnt;
  r.W0 = W0;
  dd_wave_sync();
  const unsigned long long below = (1ull << lane) - 1;
  const int n = min(nb - W0, kWindow);
  int run = 0;
  for (int j0 = 0; j0 < n; j0 += 64) {
    const int j = j0 + lane, J = W0 + j;
    bool keep = j < n, core = true;
    if (keep && J != I) {
      const unsigned bLo[3] = {lo[3 * j], lo[3 * j + 1], lo[3 * j + 2]};
      const unsigned bHi[3] = {hi[3 * j], hi[3 * j + 1], hi[3 * j + 2]};
      keep = dd_close(d, aLo, aHi, bLo, bHi, core);
    }
    const unsigned long long m = __ballot(keep);
    if (keep) {
      const int q = r.base + run + __popcll(m & below);
      if (core) atomicAdd(&r.core[min(q / d.tchunk, kRowChunks - 1)], 1);
      tile(q, J);
    }
    if (lane == 0) {
      r.bits[j0 >> 6] = m;
      r.pre[j0 >> 6] = run;
      r.ebits[j0 >> 6] = 0;
    }
    run += __popcll(m);
  }
  r.cnt = run;
  dd_wave_sync();
  dd_exclusions(d, I, [&](int sb) {
    const int q = r.place(sb / kBlockAtoms);
    if (q >= 0) atomicOr(&r.ebits[q >> 6], 1ull << (q & 63));
  });
  dd_wave_sync();
}

// one wave per i-block: its tiles, those with exclusions and its long chunks
__device__ __forceinline__ void dd_tile_count_body(const Dev &d, int bid) {
  if (halted_wg(d)) return;   // a halted step leaves the list as it is
  __shared__ __attribute__((aligned(16))) unsigned s_lo[3 * kWindow], s_hi[3 * kWindow];
  __shared__ DdRowLds s_row;
  const int nb = *d.nblocks;
  if (bid * kRows >= nb) return;
  const int w = threadIdx.x >> 6, I = bid * kRows + w, lane = threadIdx.x & 63;
  DdRow r(s_row, w);
  int flagged = 0;
  for (int W0 = 0; W0 < nb; W0 += kWindow) {
    dd_stage_boxes(d, W0, nb, s_lo, s_hi);
    if (I >= nb) continue;   // (the wave stages and waits with the others)
    dd_scan_row(d, s_lo, s_hi, W0, nb, I, r, [](int, int) {});
    for (int k = 0; 64 * k < r.cnt; k++) flagged += __popcll(r.ebits[k]);
  }
  if (I >= nb) return;
  const int cnt = r.base + r.cnt, nchunk = (cnt + d.tchunk - 1) / d.tchunk;
  int lng = 0;
  for (int k0 = 0; k0 < nchunk; k0 += 64) lng += __popcll(__ballot(k0 + lane < nchunk && r.is_long(d, k0 + lane)));
  if (lane == 0) d.rowcount[I] = make_int4(cnt, nchunk, flagged, lng);
}
__global__ void __launch_bounds__(256) dd_tile_count(Dev d) { dd_tile_count_body(d, blockIdx.x); }
__global__ void __launch_bounds__(256) dd_tile_count_multi(Multi m) {
  const MultiBlk b = multi_block(m);
  const Dev d = m.devs[b.sys];
  dd_tile_count_body(d, b.bid);
}

// One wave per row I: row starts of tiles, chunks, masks and long chunks
// (sums of the counts of the rows before: claims on shared counters instead
// serialise, 58 us at 740 rows and 200 at 2,900; flags a list that outgrows
// its buffers), then the row's tiles and chunks, and the 32 mask words of
// its tiles with exclusions (bit j of word i: slots (I,i) and (J,j) are
// excluded; tile_ex: their index, -1 for the other tiles).  No other wave
// touches the masks of the row.
__device__ __forceinline__ void dd_tile_write_body(const Dev &d, int bid) {
  if (halted_wg(d)) return;   // a halted step leaves the list as it is
  __shared__ __attribute__((aligned(16))) unsigned s_lo[3 * kWindow], s_hi[3 * kWindow];
  __shared__ DdRowLds s_row;
  __shared__ int s_sum[4 * 8];
  constexpr int kMaskTiles = 16;
  __shared__ unsigned s_mask[kRows][kMaskTiles * kBlockAtoms];
  const int nb = *d.nblocks, I0 = bid * kRows;
  if (I0 >= nb) return;
  // tiles, chunks, masks, long chunks of all rows and of the rows before
  // (32-bit sums: a list of 2^31 tiles is beyond any capacity of its arrays)
  int v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int k = threadIdx.x; k < nb; k += blockDim.x) {
    const int4 c = d.rowcount[k];
    v[0] += c.x;
    v[1] += c.y;
    v[2] += c.z;
    v[3] += c.w;
    if (k < I0) {
      v[4] += c.x;
      v[5] += c.y;
      v[6] += c.z;
      v[7] += c.w;
    }
  }
  wg_sum256(v, s_sum);
  const bool over = v[0] > d.maxtiles || v[1] > d.maxchunks;
  if (bid == 0 && threadIdx.x == 0) {
    *d.ntiles = v[0];
    *d.nchunks = v[1];
    *d.nexcltiles = v[2];
    if (over) atomicOr(d.errflag, 4);
  }
  if (over) return;
  const int w = threadIdx.x >> 6, I = I0 + w, lane = threadIdx.x & 63;
  int t0 = v[4], c0 = v[5], e = v[6], l0 = v[7];
  for (int k = I0; k < min(I, nb); k++) {
    const int4 c = d.rowcount[k];
    t0 += c.x;
    c0 += c.y;
    e += c.z;
    l0 += c.w;
  }
  DdRow r(s_row, w);
  const unsigned long long below = (1ull << lane) - 1;
  for (int W0 = 0; W0 < nb; W0 += kWindow) {
    dd_stage_boxes(d, W0, nb, s_lo, s_hi);
    if (I >= nb) continue;   // (the wave stages and waits with the others)
    dd_scan_row(d, s_lo, s_hi, W0, nb, I, r, [&](int q, int J) {
      d.tile_i[t0 + q] = I;
      d.tile_j[t0 + q] = J;
    });
    const int e0 = e;
    for (int k = 0; 64 * k < r.cnt; k++) {
      const unsigned long long m = r.ebits[k];
      const int q = k * 64 + lane;
      if (q < r.cnt) d.tile_ex[t0 + r.base + q] = (m >> lane) & 1ull ? e + __popcll(m & below) : -1;
      e += __popcll(m);
    }
    // the masks, built in LDS some tiles at a time and stored whole (clearing
    // them in memory and setting bits there takes a device-wide fence
    // between, 25 us here)
    unsigned *mask = s_mask[w];
    for (int m0 = e0; m0 < e; m0 += kMaskTiles) {
      const int words = min(kMaskTiles, e - m0) * kBlockAtoms;
      for (int k = lane; k < words; k += 64) mask[k] = 0u;
      dd_wave_sync();
      dd_exclusions(d, I, [&](int sb) {
        const int q = r.place(sb / kBlockAtoms);
        if (q < 0) return;
        int at = e0 - m0 + __popcll(r.ebits[q >> 6] & ((1ull << (q & 63)) - 1));
        for (int i = 0; i < q >> 6; i++) at += __popcll(r.ebits[i]);
        if (at >= 0 && at < kMaskTiles)
          atomicOr(&mask[at * kBlockAtoms + (lane & (kBlockAtoms - 1))], 1u << (sb % kBlockAtoms));
      });
      dd_wave_sync();
      for (int k = lane; k < words; k += 64) d.emask[(long long)m0 * kBlockAtoms + k] = mask[k];
      dd_wave_sync();
    }
  }
  if (I >= nb) return;
  const int cnt = r.base + r.cnt, tc = d.tchunk, nchunk = (cnt + tc - 1) / tc;
  if (lane == 0) {
    d.tstart[I] = t0;
    d.cstart[I] = c0;
    if (I == nb - 1) {
      d.tstart[nb] = t0 + cnt;
      d.cstart[nb] = c0 + nchunk;
    }
  }
  // The chunks, and the order of the pair kernel's waves: first the long
  // chunks.  A SIMD serves about eight waves of 2 to 16 near tiles at this
  // list's usual sizes, so the last ones to start should be short.
  int nl = l0, ns = v[3] + c0 - l0;
  for (int k0 = 0; k0 < nchunk; k0 += 64) {
    const int k = k0 + lane;
    const bool in = k < nchunk, lng = in && r.is_long(d, k);
    const unsigned long long ml = __ballot(lng), ms = __ballot(in && !lng);
    if (in) {
      d.chunk[c0 + k] = make_int4(I, t0 + k * tc, min(tc, cnt - k * tc), 0);
      d.corder[lng ? nl + __popcll(ml & below) : ns + __popcll(ms & below)] = c0 + k;
    }
    nl += __popcll(ml);
    ns += __popcll(ms);
  }
}
__global__ void __launch_bounds__(256) dd_tile_write(Dev d) { dd_tile_write_body(d, blockIdx.x); }
__global__ void __launch_bounds__(256) dd_tile_write_multi(Multi m) {
  const MultiBlk b = multi_block(m);
  const Dev d = m.devs[b.sys];
  dd_tile_write_body(d, b.bid);
}

// Every step: slot coordinates, per-block box centre/half-extent for the
// per-step cull, and reset of the force/energy accumulators.  bin: also
// the PME bins; the pack has the coordinates at hand, and a launch of their
// own at the head of the PME branch waits for CU slots behind the pair
// kernel (30 of the branch's 90 us at 23,558 atoms; 2 us here).
__device__ __forceinline__ void dd_pack_body(const Dev &d, int bid, bool bin) {
  // a halted step bins nothing (its bins would never be cleared)
  if (bin && (d.elecmethod != BM_PME || halted_wg(d))) bin = false;
  const int s = bid * blockDim.x + threadIdx.x;
  const int nb = *d.nblocks;
  const int nf = 3 * d.n + d.nl;
  if (s < nf) d.force[s] = 0;
  if (s < d.nl) {
    d.dudl[s] = 0;
    d.dtheta[s] = 0;
  }
  if (s < BM_NTERMS) d.energy[s] = 0;
  if (s < d.ncol) d.colcount[s] = 0;   // for the next rebuild
  if (bid * (int)blockDim.x >= nb * kBlockAtoms) return;  // whole wave idle
  const bool in = s < nb * kBlockAtoms;
  const int a = in ? d.l2g[s] : -1;
  unsigned u[3] = {0, 0, 0};
  if (a >= 0) {
    for (int k = 0; k < 3; k++) {
      const double x = d.pos[k * d.n + a];
      nan_check(d, x, a);
      u[k] = frac_u32(x, d.invbox[k]);
    }
    d.spos[s] = make_uint4(u[0], u[1], u[2], __float_as_uint(d.q[a]));
    d.spar[s] = make_int2(d.type[a], d.sb[a]);
    d.slo[s] = (float)(d.qd[a] - (double)d.q[a]);
  } else if (in) {
    d.spos[s] = make_uint4(0, 0, 0, 0);
    d.spar[s] = make_int2(-1, 0);
    d.slo[s] = 0.f;
  }
  if (bin) pme_bin_atom(d, a, make_uint4(u[0], u[1], u[2], 0));
  // boxes of the block (a half wave; its slot 0 is occupied) and of its four
  // clusters: lane l takes the slot at place l of the cluster order, so
  // eight neighbouring lanes hold one cluster
  const int l = threadIdx.x & (kBlockAtoms - 1);
  const int pl = in && d.clusters ? d.sperm[s] : l;
  const bool occ = __shfl(a, pl, 32) >= 0;
  int alch = (a >= 0 && d.sb[a] != 0) ? 1 : 0;
  alch = __shfl(alch, pl, 32);
  for (int o = 4; o > 0; o >>= 1) alch |= __shfl_xor(alch, o, 32);
  const int calch = alch;
  for (int o = 16; o > 4; o >>= 1) alch |= __shfl_xor(alch, o, 32);
  const unsigned long long om = __ballot(occ);
  const bool cocc = (om >> (threadIdx.x & 56)) & 0xFFull;
  unsigned c[3], h[3], cc[3];
  float ch[3];
  for (int k = 0; k < 3; k++) {
    const unsigned ref = __shfl(u[k], 0, 32);
    const int off = __shfl((int)(u[k] - ref), pl, 32);
    int mn = occ ? off : 0x7FFFFFFF, mx = occ ? off : (int)0x80000000;
    for (int o = 4; o > 0; o >>= 1) {
      mn = min(mn, __shfl_xor(mn, o, 32));
      mx = max(mx, __shfl_xor(mx, o, 32));
    }
    // (mn + mx may pass 2^31: slot 0 need not be in the cluster)
    cc[k] = cocc ? ref + (unsigned)mn + ((unsigned)(mx - mn) >> 1) : ref;
    ch[k] = cocc ? (float)((unsigned)(mx - mn + 1) >> 1) * d.fracscale[k] : -1e15f;
    for (int o = 16; o > 4; o >>= 1) {
      mn = min(mn, __shfl_xor(mn, o, 32));
      mx = max(mx, __shfl_xor(mx, o, 32));
    }
    c[k] = ref + (unsigned)((mn + mx) >> 1);
    h[k] = (unsigned)(mx - mn + 1) >> 1;
  }
  if (in && d.clusters && (s & (kClusterAtoms - 1)) == 0) {
    d.sbc[s / kClusterAtoms] = make_uint4(cc[0], cc[1], cc[2], (unsigned)calch);
    d.sbh[s / kClusterAtoms] = make_float4(ch[0], ch[1], ch[2], 0.f);
  }
  if (in && (s & (kBlockAtoms - 1)) == 0) {
    const int b = s / kBlockAtoms;
    d.bbc[b] = make_uint4(c[0], c[1], c[2], 0);
    d.bbh[b] = make_uint4(h[0], h[1], h[2], (unsigned)alch);
  }
}

__global__ void __launch_bounds__(256) dd_pack(Dev d, bool bin) { dd_pack_body(d, blockIdx.x, bin); }

__global__ void __launch_bounds__(256) dd_pack_multi(Multi m) {
  const MultiBlk b = multi_block(m);
  const Dev d = m.devs[b.sys];
  dd_pack_body(d, b.bid, true);
}

// ---------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------
void launch_domdec_rebuild(const Dev &d, int maxBlocks, hipStream_t st) {
  (void)maxBlocks;
  dd_wrap_count<<<grid_rebuild(d, 0), 256, 0, st>>>(d);
  if (grid_rebuild(d, 1)) dd_scan_columns<<<1, 256, 0, st>>>(d);
  dd_scatter<<<grid_rebuild(d, 2), 256, 0, st>>>(d);
  dd_sort_columns<<<grid_rebuild(d, 3), 256, 0, st>>>(d);
  dd_tile_count<<<grid_rebuild(d, 4), 256, 0, st>>>(d);
  dd_tile_write<<<grid_rebuild(d, 5), 256, 0, st>>>(d);
}

// The rebuild's kernels in order, for one launch each over several systems:
// workgroups of kernel k for system d (0 leaves d out of that launch), and the
// launches over the per-kernel plans m[kRebuildKernels].
int grid_rebuild(const Dev &d, int k) {
  const int slots = (int)((32LL * d.maxblocks + 255) / 256), rows = (d.maxblocks + kRows - 1) / kRows;
  switch (k) {
    case 0: return slots;                // dd_wrap_count
    case 1: return d.ncol > kScanCols;   // dd_scan_columns
    case 2: return slots;                // dd_scatter
    case 3: return d.ncol;               // dd_sort_columns
    default: return rows;                // dd_tile_count, dd_tile_write: a wave per block
  }
}

void launch_domdec_rebuild_multi(const Multi *m, hipStream_t st) {
  dd_wrap_count_multi<<<m[0].nwg, 256, 0, st>>>(m[0]);
  if (m[1].nwg) dd_scan_columns_multi<<<m[1].nwg, 256, 0, st>>>(m[1]);
  dd_scatter_multi<<<m[2].nwg, 256, 0, st>>>(m[2]);
  dd_sort_columns_multi<<<m[3].nwg, 256, 0, st>>>(m[3]);
  dd_tile_count_multi<<<m[4].nwg, 256, 0, st>>>(m[4]);
  dd_tile_write_multi<<<m[5].nwg, 256, 0, st>>>(m[5]);
}

int grid_pack(const Dev &d) {
  long long work = (long long)d.maxblocks * kBlockAtoms;
  long long nf = 3LL * d.n + d.nl;
  if (nf > work) work = nf;
  if (work < BM_NTERMS) work = BM_NTERMS;
  return (int)((work + 255) / 256);
}

void launch_domdec_pack(const Dev &d, int maxBlocks, hipStream_t st, bool bin) {
  (void)maxBlocks;
  dd_pack<<<grid_pack(d), 256, 0, st>>>(d, bin);
}

void launch_pack_multi(const Multi &m, hipStream_t st) { dd_pack_multi<<<m.nwg, 256, 0, st>>>(m); }

}  // namespace blade
