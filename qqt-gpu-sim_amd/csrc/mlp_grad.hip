// First-layer weight gradient of the mlp ActorCritic for the PPO update
// (train/ppo.py:364-437 runs loss.backward() through train/model.py:121-147):
//   dW0[h][k] = sum_b dz1[b][h] * obs[b][k]
// over a minibatch of B observation rows (float16, exact) and the float32
// gradient dz1 of the first layer's output.  This product carries nearly all
// of the backward pass's work and bytes (K = 2366 observation columns per
// row; the later layers are 128 wide).
//
// MFMA v_mfma_f32_16x16x32_f16 with the batch as the contraction index.  The
// observation is exact in float16; dz1 is scaled by a power of two (so its
// largest magnitude is 2^14) and split into float16 hi + lo, two products per
// tile, which keeps the result within ~1e-6 relative of a float32 sum.
//
// Grid: (column tile of 512 observation columns) x (chunk of the batch); tiles of
// 128 columns where the workspace has slots for groups of chunks only (Plan) or
// the grid is small (l1_grad_launch).  A
// workgroup (8 wavefronts, one per CU) owns a 128 x 512 float32 output tile
// for its chunk, 64 x 128 per wavefront in registers, and walks the chunk 32
// rows at a time.  Each step's 32 KB of observation and 16 KB of dz1 are
// loaded two steps ahead into registers and stored to LDS as they are, row by
// row (dz1 as hi and lo planes); the MFMA operands, which need the batch index
// contiguous per lane, are read through the transposing ds_read_b64_tr_b16.
// One barrier per step.  Partial tiles go to a workspace
// [slot][128][tiles * width]; a second kernel sums the slots in a fixed order
// (deterministic) and applies the inverse scale.
//
// Bound: HBM, 2 k0 + 512 bytes per row (the observation once; dz1 once per
// column tile, the repeats from the caches), beside 128 k0 multiply-adds per
// row in two products.  Tiles of 256 columns (two workgroups per CU) read and
// split dz1 twice as often, transposed both operands with VALU permutes and
// had one step of loads in flight: a 180,224-row minibatch of scattered rows
// took 335 us, now 280; with its rows cached 231 (a library float16 product of
// 8192^3 reaches 1.2 PFLOP/s on the same card: 180 us).

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <mutex>
#include <type_traits>

#include "mlp_common.h"
#include "qqt_common.h"
#include "qqt_hip.h"
#include "qqt_learn.h"

namespace qqt {

extern thread_local char g_err[512];

namespace l1g {

constexpr int NCOL = 512;         // observation columns per workgroup ...
constexpr int NARROW = 128;       // ... and where its slot takes several chunks or the grid is small
constexpr int KS = 32;            // batch rows per step (one MFMA K)
// LDS row strides (halves; NC + 16 for the observation), 8 banks apart per row:
// 16-byte stores and the transposing reads (4 rows of 32 bytes per 16 lanes)
// are conflict-free
constexpr int DS = HID + 16;
constexpr int NT = 512;           // threads
constexpr int MAX_CHUNKS = 64;
constexpr int TARGET_WGS = 256;   // one workgroup (104 KB of LDS, 256 registers) per CU
constexpr int CHUNK_ROWS = 512;   // least rows of a chunk
constexpr int SLOT_ROWS = 2048;   // ... of a slot of the workspace every caller provides

template <int NC>
struct __align__(16) Lds {
  uint16_t x[2][KS][NC + 16];     // observation rows
  uint16_t d[2][2][KS][DS];       // dz1 rows, hi and lo planes
};

// Accumulators of a wavefront: four m tiles x JT n tiles.
template <int NC>
struct Tile {
  static constexpr int JT = NC / 64;
  floatx4 v[4][JT];
};

// One chunk's product for a tile of NC columns, from zero.
// EDGE: the tile reaches past column k0 (or its rows are shorter than a
// 16-byte chunk): loads go dword by dword, clamped into the row; columns at
// or past k0 hold repeats that only reach output columns nobody reads.
template <int NC, bool EDGE>
__device__ __forceinline__ void l1_grad_chunk(const qqt_l1_grad_args& a, Lds<NC>& s, int tile,
                                              int chunk, int chunk_rows, Tile<NC>& acc) {
  constexpr int XS = NC + 16, JT = Tile<NC>::JT;
  constexpr int LPR = NC / 8;             // lanes of an observation row (16 bytes each)
  constexpr int RPL = 64 / LPR, NL = 4 / RPL;    // rows per load, loads per step
  const int t = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const int col0 = tile * NC;
  const int r_begin = chunk * chunk_rows;
  const int r_end = min(r_begin + chunk_rows, a.batch);
  const int steps = (r_end - r_begin + KS - 1) / KS;     // >= 1 (chunks are non-empty)
  const float scale = a.dz_scale ? *a.dz_scale : 1.0f;

  // loader roles: wavefront w brings rows 4w .. 4w + 3 of the observation,
  // lane l columns 8 (l % LPR) .. + 7 of row l / LPR of each load; thread t row
  // t / 16 of dz1, hidden 8 (t % 16) .. + 7.  Rows past the chunk load its last
  // row again and are stored as zeros on both sides (an infinity or NaN of that
  // row against a zero gradient would be NaN).
  const int dr = t >> 4, dc = 8 * (t & 15);
  struct Regs {
    u32x4 x[NL];
    float d[8];
  };
  // Rows of the wavefront in a step: lane l holds the buffer row of row
  // 4w + l % 4, loaded a step before the observation rows it points at (and
  // before that step's loads, so waiting for it waits for nothing younger).
  int64_t at;
  auto index = [&](int step) {
    const int r = min(r_begin + KS * step + 4 * w + (lane & 3), r_end - 1);
    at = a.row_index ? a.row_index[r] : (int64_t)r;
  };
  auto load = [&](int step, Regs& g) {
    const int r0 = r_begin + KS * step;
    const int64_t row = a.row_index ? min(max(at, (int64_t)0), a.obs_rows - 1) : at;
    const int lo = (int)row, hi = (int)(row >> 32);
    index(min(step + 1, steps - 1));
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      uint32_t rl, rh;
      if constexpr (RPL == 1) {
        rl = __builtin_amdgcn_readlane(lo, i);
        rh = __builtin_amdgcn_readlane(hi, i);
      } else {
        rl = __shfl(lo, RPL * i + lane / LPR, 64);
        rh = __shfl(hi, RPL * i + lane / LPR, 64);
      }
      const int64_t ri = (int64_t)(((uint64_t)rh << 32) | rl);
      const uint16_t* const p = a.obs + ri * a.obs_stride;
      const int c = 8 * (lane % LPR);
      if constexpr (EDGE) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          g.x[i][k] = reinterpret_cast<const uint32_t*>(p)[min(((col0 + c) >> 1) + k, (a.k0 >> 1) - 1)];
      } else {
        __builtin_memcpy(&g.x[i], p + col0 + c, 16);             // 4-byte aligned
      }
    }
    __builtin_memcpy(g.d, a.dz1 + (size_t)min(r0 + dr, r_end - 1) * HID + dc, 32);
  };
  // (end: the step may reach past the chunk)
  auto store = [&](const Regs& g, int buf, int step, auto end) {
    const int r0 = r_begin + KS * step;
    const bool live = !decltype(end)::value || r0 + dr < r_end;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int r = 4 * w + RPL * i + lane / LPR;
      u32x4 x = g.x[i];
      if (decltype(end)::value && r0 + r >= r_end) x = u32x4{0, 0, 0, 0};
      *reinterpret_cast<u32x4*>(&s.x[buf][r][8 * (lane % LPR)]) = x;
    }
    half8 hi, lo;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float v = live ? g.d[k] * scale : 0.0f;
      hi[k] = (_Float16)v;
      lo[k] = (_Float16)(v - (float)hi[k]);
    }
    *reinterpret_cast<half8*>(&s.d[buf][0][dr][dc]) = hi;
    *reinterpret_cast<half8*>(&s.d[buf][1][dr][dc]) = lo;
  };

  // wavefront w: hidden 64 (w & 1) .. + 63 (four m tiles), column quarter w / 2
  const int mt = 4 * (w & 1), nt = JT * (w >> 1);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j) acc.v[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  auto compute = [&](int buf) {
    if constexpr (NC == NARROW) {       // few n tiles: hold those, pass the m tiles through
      half8 b[JT];
#pragma unroll
      for (int j = 0; j < JT; ++j) b[j] = ld_rows<half8, XS>(&s.x[buf][0][0], nt + j, lane);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const half8 ah = ld_rows<half8, DS>(&s.d[buf][0][0][0], mt + i, lane);
        const half8 al = ld_rows<half8, DS>(&s.d[buf][1][0][0], mt + i, lane);
#pragma unroll
        for (int j = 0; j < JT; ++j) acc.v[i][j] = mfma(ah, b[j], acc.v[i][j]);
#pragma unroll
        for (int j = 0; j < JT; ++j) acc.v[i][j] = mfma(al, b[j], acc.v[i][j]);
      }
    } else {
      half8 ah[4], al[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ah[i] = ld_rows<half8, DS>(&s.d[buf][0][0][0], mt + i, lane);
        al[i] = ld_rows<half8, DS>(&s.d[buf][1][0][0], mt + i, lane);
      }
#pragma unroll
      for (int j = 0; j < JT; ++j) {
        const half8 b = ld_rows<half8, XS>(&s.x[buf][0][0], nt + j, lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc.v[i][j] = mfma(ah[i], b, acc.v[i][j]);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc.v[i][j] = mfma(al[i], b, acc.v[i][j]);
      }
    }
  };

  // Register ring of two steps in flight beside the LDS double buffer: step i
  // computes from buffer i & 1, stores step i + 1 to the other and loads step
  // i + 3 into the slot that freed (steps past the last reload the last).
  // Only the last step can reach past the chunk, and it is not stored in the loop.
  Regs g[2];
  const int last = steps - 1;
  const std::integral_constant<bool, true> may_end;
  const std::integral_constant<bool, false> whole;
  index(0);
  load(0, g[0]);
  load(min(1, last), g[1]);
  store(g[0], 0, 0, may_end);
  load(min(2, last), g[0]);
  __syncthreads();
  int i = 0;
  for (; i + 2 < last; i += 2) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      compute(k);
      store(g[1 - k], 1 - k, i + k + 1, whole);
      load(min(i + k + 3, last), g[1 - k]);
      __syncthreads();
    }
  }
  compute(0);
  if (i < last) {
    store(g[1], 1, i + 1, may_end);
    __syncthreads();
    compute(1);
    if (i + 1 < last) {
      store(g[0], 0, last, may_end);
      __syncthreads();
      compute(0);
    }
  }
}

// Column tile blockIdx.x of slot blockIdx.y -> workspace [slot][hidden][ws_cols].
// A slot takes one chunk in the wide tile; in the narrow one up to `per_slot`
// consecutive chunks, their products added in order in registers.
// (Dealing the column tiles of a chunk to one XCD, so that its L2 serves dz1
// to all of them, leaves 240 of the 256 CUs at work and measured 308 us
// against 294; tiles of 256 columns, two workgroups per CU, 317 us.  Adding a
// slot's chunks in the workspace instead, which the wide tile would need, took
// 232 us for 8,192 rows in four slots.)  The narrow tile is held to 128 registers
// (7 go to scratch): two workgroups per CU take 45,056 rows in 17 slots in
// 114 us, one (156 registers) in 134.
template <int NC, bool EDGE>
__device__ __forceinline__ void l1_grad_slot(const qqt_l1_grad_args& a, Lds<NC>& s, int chunks,
                                             int chunk_rows, int ws_cols, int per_slot) {
  constexpr int JT = Tile<NC>::JT;
  Tile<NC> sum;
  if constexpr (NC == NARROW) {
    const int first = blockIdx.y * per_slot, end = min(first + per_slot, chunks);
#pragma unroll 1
    for (int c = first; c < end; ++c) {
      Tile<NC> acc;
      l1_grad_chunk<NC, EDGE>(a, s, blockIdx.x, c, chunk_rows, acc);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j) sum.v[i][j] = c == first ? acc.v[i][j] : sum.v[i][j] + acc.v[i][j];
      __syncthreads();                  // every wavefront is done with this chunk's LDS
    }
  } else {
    l1_grad_chunk<NC, EDGE>(a, s, blockIdx.x, blockIdx.y, chunk_rows, sum);
  }
  // lane holds hidden rows 4(lane/16)+q of each m tile at column lane%16 of each n tile
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int mt = 4 * (w & 1), nt = JT * (w >> 1);
  float* const out = a.workspace + (size_t)blockIdx.y * HID * ws_cols + blockIdx.x * NC;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        out[(size_t)(16 * (mt + i) + 4 * (lane >> 4) + q) * ws_cols + 16 * (nt + j) + (lane & 15)] = sum.v[i][j][q];
}

template <int NC>
__global__ __launch_bounds__(NT, NC == NARROW ? 4 : 2) void l1_grad_kernel(
    const qqt_l1_grad_args a, int chunks, int chunk_rows, int ws_cols, int per_slot) {
  __shared__ Lds<NC> s;
  if ((int)(blockIdx.x + 1) * NC <= a.k0)
    l1_grad_slot<NC, false>(a, s, chunks, chunk_rows, ws_cols, per_slot);
  else
    l1_grad_slot<NC, true>(a, s, chunks, chunk_rows, ws_cols, per_slot);
}

// dw0[h][cols ? cols[k] : k] = (sum over groups of `group` slots, in order, each
// the sum of its slots in order) / scale, k < k0.  A column index outside
// [0, k0) is clamped into it.  Bound: HBM and the Infinity Cache (51 partials
// of 1.3 MB for a 180,224-row minibatch); eight loads in flight per thread.
__global__ __launch_bounds__(256) void l1_grad_reduce(const qqt_l1_grad_args a, int slots, int group,
                                                      int ws_cols, const int64_t* cols) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= HID * a.k0) return;
  const int h = i / a.k0, k = i % a.k0;
  const float inv = a.dz_scale ? 1.0f / *a.dz_scale : 1.0f;   // power of two: exact
  const size_t pitch = (size_t)HID * ws_cols;
  const float* p = a.workspace + (size_t)h * ws_cols + k;
  const int64_t col = cols ? min(max(cols[k], (int64_t)0), (int64_t)a.k0 - 1) : (int64_t)k;
  float sum = 0.0f, part = 0.0f;
  int at = 0, c = 0;                  // at: slots that the current group has taken
  auto add = [&](float v) {
    part = at == 0 ? v : part + v;
    if (++at == group) {
      sum += part;
      at = 0;
    }
  };
  for (; c + 8 <= slots; c += 8, p += 8 * pitch) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = p[j * pitch];
#pragma unroll
    for (int j = 0; j < 8; ++j) add(v[j]);
  }
  for (; c < slots; ++c, p += pitch) add(*p);
  if (at) sum += part;
  a.dw0[(size_t)h * a.k0 + col] = sum * inv;
}

// The first layer's weight as the float16 MFMA B fragments the forward reads,
// [tile][kblock][lane 16 q + r][16]: value i is row 16 tile + r, column
// cols[64 kblock + 16 q + i], zero from k0 on.  A thread writes 16 bytes; a
// launch moves 1.8 MB (1.2 read, 0.6 written) and is latency (5 us).  In its
// place were an index, a fill, two copies and a conversion; with the column
// order of dW0 (another index launch) folded into l1_grad_reduce, 33 us of the
// gradients of an 8192-row minibatch (192 -> 159) and 29 of 180,224 rows.
__global__ __launch_bounds__(256) void w0_pack_kernel(const float* w, const int64_t* cols, int k0,
                                                      int kblocks, uint16_t* out) {
  const int i = blockIdx.x * 256 + threadIdx.x;           // 8 halves each
  if (i >= HID / 16 * kblocks * 128) return;
  const int lane = (i >> 1) & 63, kb = (i >> 7) % kblocks, tile = (i >> 7) / kblocks;
  const int k = 64 * kb + 16 * (lane >> 4) + 8 * (i & 1);
  const float* const row = w + (size_t)(16 * tile + (lane & 15)) * k0;
  half8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int64_t col = k + j < k0 ? min(max(cols[k + j], (int64_t)0), (int64_t)k0 - 1) : 0;
    v[j] = k + j < k0 ? (_Float16)row[col] : (_Float16)0.0f;
  }
  *reinterpret_cast<half8*>(out + 8 * (size_t)i) = v;
}

// Pieces of the batch: rows of each a multiple of KS, at least min_rows, and
// pieces x column tiles at most TARGET_WGS (all workgroups resident at once,
// one per CU) and MAX_CHUNKS: a 180,224-row minibatch of 2366 columns makes 51
// pieces x 5 tiles.
__host__ inline int pieces(int batch, int k0, int min_rows, int& rows) {
  const int tiles = (k0 + NCOL - 1) / NCOL;
  int n = (batch - 1) / min_rows + 1;
  if (n > TARGET_WGS / tiles) n = TARGET_WGS / tiles;
  if (n > MAX_CHUNKS) n = MAX_CHUNKS;
  if (n < 1) n = 1;
  rows = (batch - 1) / n + 1;
  rows = (rows - 1) / KS * KS + KS;
  return (batch - 1) / rows + 1;
}

// The order of the sums follows the batch and k0 alone: chunks of at least
// CHUNK_ROWS rows, each a product of its own; groups of consecutive chunks,
// each summed in chunk order; the groups summed in order.  There are at most as
// many groups as the documented workspace (SLOT_ROWS) has slots.  A workspace
// that holds every chunk's partial gives each chunk its own workgroups and
// leaves both sums to the reduction; in a smaller one a slot's workgroups, of
// the narrow tile, walk its group's chunks and add as they go.  Below 512 rows a
// chunk's partial tiles (1.3 MB out and back) cost what the shorter walk saves.
// With the reduction, 2366 columns, in the documented workspace (one chunk per
// slot, wide tile -> groups) and in the preferred one: 8,192 rows 134 -> 58 and
// 32 us, 45,056 rows 142 -> 114 and 90 us.
struct Plan {
  int chunks, rows, group;
};
__host__ inline Plan plan(int batch, int k0) {
  Plan p;
  int slot_rows;
  const int slots = pieces(batch, k0, SLOT_ROWS, slot_rows);
  p.chunks = pieces(batch, k0, CHUNK_ROWS, p.rows);
  if (p.chunks <= slots + slots / 8) {     // a few chunks more are not worth walking
    p.chunks = slots;
    p.rows = slot_rows;
  }
  p.group = (p.chunks + slots - 1) / slots;
  return p;
}

__host__ inline int64_t slot_floats(int k0) {
  return (int64_t)HID * ((k0 + NCOL - 1) / NCOL) * NCOL;
}

}  // namespace l1g

// Scratch of qqt_l1_grad_noalloc: the chunk partials of the largest plan
// (MAX_CHUNKS chunks of 128 x QQT_L1_GRAD_NOALLOC_MAX_K0 columns), one copy
// per GPU, held until the process ends.  Host code never passes this name
// to a kernel (on the host it is only a stand-in for the symbol): it uses
// the device address hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) float
    l1g_scratch[l1g::MAX_CHUNKS * HID * QQT_L1_GRAD_NOALLOC_MAX_K0];

namespace l1g {

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[MAX_DEVICES] = {};

// The scratch's device address on the current device, looked up once per
// device (with that device current); nullptr with g_err set on failure.
float* scratch_on_current_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
    snprintf(g_err, sizeof(g_err), "qqt_l1_grad_noalloc: no usable current device");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(l1g_scratch));
    if (err != hipSuccess || !p) {
      snprintf(g_err, sizeof(g_err), "qqt_l1_grad_noalloc: hipGetSymbolAddress failed: %s",
               hipGetErrorString(err));
      return nullptr;
    }
    g_scratch_ptr[dev] = static_cast<float*>(p);
  }
  return g_scratch_ptr[dev];
}

}  // namespace l1g
}  // namespace qqt

extern "C" {

int64_t qqt_l1_grad_workspace_floats(int32_t batch, int32_t k0) {
  using namespace qqt::l1g;
  if (batch <= 0 || k0 <= 0) return -1;
  int rows;
  return pieces(batch, k0, SLOT_ROWS, rows) * slot_floats(k0);
}

int64_t qqt_l1_grad_preferred_floats(int32_t batch, int32_t k0) {
  using namespace qqt::l1g;
  if (batch <= 0 || k0 <= 0) return -1;
  return plan(batch, k0).chunks * slot_floats(k0);
}

namespace {

// Shape checks shared by both entry points (the workspace is checked by the
// caller of each).
int l1_grad_check(const qqt_l1_grad_args* a, const char* who) {
  using namespace qqt;
  if (!a || !a->obs || !a->dz1 || !a->dw0) {
    snprintf(g_err, sizeof(g_err), "%s: null argument", who);
    return QQT_E_ARG;
  }
  if (a->batch <= 0 || a->k0 <= 0 || (a->k0 & 1) || a->obs_stride < a->k0 ||
      (a->obs_stride & 1) || (((uintptr_t)a->obs) & 3) || (((uintptr_t)a->dz1) & 7)) {
    snprintf(g_err, sizeof(g_err), "%s: bad shape/stride/alignment", who);
    return QQT_E_ARG;
  }
  if (a->row_index && (a->obs_rows <= 0 || (((uintptr_t)a->row_index) & 7))) {
    snprintf(g_err, sizeof(g_err), "%s: row_index needs obs_rows > 0 and 8-byte alignment", who);
    return QQT_E_ARG;
  }
  return QQT_OK;
}

int l1_grad_workspace_check(const qqt_l1_grad_args& a, const char* who) {
  using namespace qqt;
  if (!a.workspace) {
    snprintf(g_err, sizeof(g_err), "%s: null workspace", who);
    return QQT_E_ARG;
  }
  if (a.workspace_floats < qqt_l1_grad_workspace_floats(a.batch, a.k0)) {
    snprintf(g_err, sizeof(g_err), "%s: workspace too small", who);
    return QQT_E_ARG;
  }
  return QQT_OK;
}

// Both launches over a checked argument block whose workspace holds the
// plan's partials.
int l1_grad_launch(const qqt_l1_grad_args& a, hipStream_t st, const int64_t* cols = nullptr) {
  using namespace qqt;
  using namespace qqt::l1g;
  const Plan p = plan(a.batch, a.k0);
  const bool whole = a.workspace_floats >= p.chunks * slot_floats(a.k0);
  const int per_slot = whole ? 1 : p.group;
  const int slots = (p.chunks - 1) / per_slot + 1;
  // The narrow tile also where the wide ones would leave three eighths of the
  // CUs idle: a step of 32 rows takes a workgroup of the wide tile four times
  // the products.  Wide and narrow, with the reduction, in the preferred
  // workspace: 2366 columns, 1 row 11.4 and 7.4 us, 512 rows (5 wide tiles) 39
  // and 18, 8,192 (80) 45 and 32, 20,000 (200) 52 and 55, 45,056 (255) 90 and
  // 101; 686 columns, 45,056 rows (128) 55 and 49, 180,224 (128) 187 and 151.
  const bool narrow = per_slot > 1 || (a.k0 + NCOL - 1) / NCOL * slots * 8 <= TARGET_WGS * 5;
  const int ncol = narrow ? NARROW : NCOL;
  const int tiles = (a.k0 + ncol - 1) / ncol, ws_cols = tiles * ncol;
  if (narrow)
    QQT_LAUNCH(QQT_KERNEL_L1GRAD, l1_grad_kernel<NARROW>, dim3(tiles, slots), dim3(NT), st, a,
               p.chunks, p.rows, ws_cols, per_slot);
  else
    QQT_LAUNCH(QQT_KERNEL_L1GRAD, l1_grad_kernel<NCOL>, dim3(tiles, slots), dim3(NT), st, a,
               p.chunks, p.rows, ws_cols, per_slot);
  hipError_t err = hipGetLastError();
  if (err == hipSuccess) {
    const int n = HID * a.k0;
    QQT_LAUNCH(QQT_KERNEL_L1GRAD, l1_grad_reduce, dim3((n + 255) / 256), dim3(256), st, a,
               slots, whole ? p.group : 1, ws_cols, cols);
    err = hipGetLastError();
  }
  if (err != hipSuccess) {
    snprintf(g_err, sizeof(g_err), "l1 grad launch failed: %s", hipGetErrorString(err));
    return QQT_E_LAUNCH;
  }
  return QQT_OK;
}

}  // namespace

int qqt_l1_grad(const qqt_l1_grad_args* a, void* stream) {
  using namespace qqt;
  g_err[0] = 0;
  if (const int rc = l1_grad_check(a, "qqt_l1_grad")) return rc;
  if (const int rc = l1_grad_workspace_check(*a, "qqt_l1_grad")) return rc;
  return l1_grad_launch(*a, (hipStream_t)stream);
}

int qqt_l1_grad_columns(const qqt_l1_grad_args* a, const int64_t* cols, void* stream) {
  using namespace qqt;
  g_err[0] = 0;
  if (const int rc = l1_grad_check(a, "qqt_l1_grad_columns")) return rc;
  if (const int rc = l1_grad_workspace_check(*a, "qqt_l1_grad_columns")) return rc;
  if (!cols || (((uintptr_t)cols) & 7)) {
    snprintf(g_err, sizeof(g_err), "qqt_l1_grad_columns: cols must be an 8-byte aligned device array");
    return QQT_E_ARG;
  }
  return l1_grad_launch(*a, (hipStream_t)stream, cols);
}

int qqt_w0_pack(const float* w, const int64_t* cols, int32_t k0, int32_t kblocks, void* out,
                void* stream) {
  using namespace qqt;
  using namespace qqt::l1g;
  g_err[0] = 0;
  if (!w || !cols || !out) {
    snprintf(g_err, sizeof(g_err), "qqt_w0_pack: null argument");
    return QQT_E_ARG;
  }
  if (k0 <= 0 || kblocks != (k0 - 1) / 64 + 1 || kblocks > (1 << 20) || (((uintptr_t)w) & 3) ||
      (((uintptr_t)cols) & 7) || (((uintptr_t)out) & 15)) {
    snprintf(g_err, sizeof(g_err), "qqt_w0_pack: bad k0, kblocks or alignment");
    return QQT_E_ARG;
  }
  hipLaunchKernelGGL(w0_pack_kernel, dim3(HID / 16 * kblocks * 128 / 256), dim3(256), 0,
                     (hipStream_t)stream, w, cols, k0, kblocks, static_cast<uint16_t*>(out));
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    snprintf(g_err, sizeof(g_err), "w0 pack launch failed: %s", hipGetErrorString(err));
    return QQT_E_LAUNCH;
  }
  return QQT_OK;
}

int qqt_l1_grad_noalloc(const qqt_l1_grad_args* a, void* stream) {
  using namespace qqt;
  g_err[0] = 0;
  if (const int rc = l1_grad_check(a, "qqt_l1_grad_noalloc")) return rc;
  if (a->k0 > QQT_L1_GRAD_NOALLOC_MAX_K0) {
    snprintf(g_err, sizeof(g_err),
             "qqt_l1_grad_noalloc: k0 = %d exceeds the static scratch's maximum of %d columns",
             a->k0, QQT_L1_GRAD_NOALLOC_MAX_K0);
    return QQT_E_ARG;
  }
  float* const ptr = l1g::scratch_on_current_device();
  if (!ptr) return QQT_E_LAUNCH;
  qqt_l1_grad_args b = *a;          // the caller's workspace fields are ignored
  b.workspace = ptr;
  b.workspace_floats = qqt_l1_grad_preferred_floats(b.batch, b.k0);
  if (b.workspace_floats > (int64_t)l1g::MAX_CHUNKS * HID * QQT_L1_GRAD_NOALLOC_MAX_K0) {
    snprintf(g_err, sizeof(g_err), "qqt_l1_grad_noalloc: plan exceeds the static scratch");
    return QQT_E_ARG;
  }
  return l1_grad_launch(b, (hipStream_t)stream);
}

}  // extern "C"
