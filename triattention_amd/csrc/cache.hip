// Decode-cache assembly on the device: the kept-tile metadata of one Prefill call's batch and the
// compaction of its records into the cache's arrays.
//
// Reference semantics: triattention/kernels/decode.py:24-67 (DecodeCache.store), which classifies the
// tiles and compacts the records on the host with torch.  The rules are its own:
//   * state of tile j for a q-head with band (w8, w4): 8 if j == 0 or d < w8, 4 if d < w4, else 0,
//     with d = tiles - 1 - j (decode.py:27-30);
//   * K precision of a (KV head, tile): the maximum state over the head's GQA group; the tile is kept
//     when that is > 0, and its rowmask has bit r set when q-head r of the group has state > 0
//     (decode.py:31-33);
//   * kept tiles of a head are listed in ascending order (decode.py:36); INT4 and INT8 K records, and
//     INT8 and INT4 V records, are each numbered in (KV head, entry) order (decode.py:38-53);
//   * V is INT8 for the sink tile and the last NEAR_V8 tiles, INT4 elsewhere (decode.py:17-22).
// Extension: KV heads kept exact (bf16) keep every tile with every q-head's bit set, select no quantized
// record, and copy their KX / VX records whole.
//
// Every state depends on the tile's distance from the end alone, so each head's kept, INT8-K, INT4-K, INT8-V
// and INT4-V tiles are tile 0 and runs of consecutive tiles whose ends follow from the largest w8 and w4 of
// the group: entry indices and record slots have closed forms, and no workgroup scans tiles or waits for
// another.  One workgroup per (run of tiles, KV head, sequence): it forms every head's counts (one thread
// per head), copies its tiles' records with 16-byte accesses, K and V loads in flight together, and the
// chunk-0 workgroup of a head writes the head's metadata row.  HBM-bound for many tiles, one launch's latency
// for few: against classifying and scanning every head's tiles in every workgroup and 16 tiles copied one
// after another, 64 tiles x 4 KV heads (one exact) 43.5 -> 10.3 us, one tile x 8 KV heads 12.0 -> 7.3 us,
// 64 tiles x 8 KV heads x 32 sequences 92 -> 94 us.
#include "common.h"

namespace tri {

// Tiles whose records one workgroup copies: as many as keep the launch at STORE_WGS workgroups, at most
// STORE_CHUNK (few tiles: one each, so that their latencies overlap; many: each workgroup's counts are shared by
// more copies.  At most 2 / 4 / 8 per workgroup: 256 tiles 12.6 / 17.8 / - (one: 10.1), 16,384 tiles 113 / 94 / 110 us).
constexpr int STORE_CHUNK = 4, STORE_WGS = 2048;
constexpr int STORE_THREADS = 256;
constexpr int STORE_MAX_HQ = 256;  // q-heads whose bands the kernel stages in LDS

struct CacheStoreArgs {
  const int32_t* bands;  // [hq][2] (w8, w4)
  const int32_t* exact;  // [hk]: -1 for a quantized KV head, else its slot among the exact heads; may be null
  int hq, hk, t, tiles, nx, batch, chunk;  // chunk: tiles per workgroup
  int xstride;  // records per (sequence, exact head) in the destination (>= tiles: room for tail tiles)
  // sources: the Prefill call's outputs, [batch][hk][tiles] records and scales
  const uint8_t* kp;   // K8
  const uint8_t* k4p;  // K4 (may be null when no tile is INT4)
  const uint8_t* v8p;
  const uint8_t* v4p;  // (may be null when no tile has INT4 V)
  const uint8_t* kx;   // [batch][nx][tiles] KX / VX records of the exact heads (may be null)
  const uint8_t* vx;
  const float* ka;     // [batch][hk][tiles][4]
  const float* ka4;    // (may be null)
  const float* kstat;  // [batch][hk][3][128]
  const float* vstat;
  // destination: rows row0 .. row0 + batch - 1 of the cache (rows allocated: `rows`)
  int row0, rows, maxn, tiles_max;
  int32_t* entry;  // [rows][hk][maxn]
  int32_t* kinfo;
  int32_t* slot;
  int32_t* count;  // [rows][hk]
  int32_t* fmt;    // [rows][tiles_max]
  int32_t* prompt; // [rows]
  int32_t* xslot;  // [rows][hk] (may be null when no head is exact)
  float* ka_c;     // [rows][hk][tiles_max][4]
  float* ka4_c;    // (may be null)
  float* kstat_c;  // [rows][hk][3][128]
  float* vstat_c;
  uint8_t* k8c;    // compacted record arrays, first free record o*, records held cap*
  uint8_t* k4c;
  uint8_t* v8c;
  uint8_t* v4c;
  uint8_t* kxc;
  uint8_t* vxc;
  int64_t o8, o4, ov8, ov4, ox;
  int64_t cap8, cap4, capv8, capv4, capx;
};

// A head's tile runs: kept tiles are 0 and [keep, tiles), INT8-K ones (quantized heads) 0 and [k8, tiles),
// INT4-K ones [keep, k8), INT8-V ones 0 and [v8, tiles), INT4-V ones [keep, v8).
struct HeadRuns {
  int keep, k8, v8;
};
__device__ __forceinline__ HeadRuns head_runs(const int* bands, int g, bool ex, int tiles) {
  int w8 = 0, w4 = 0;
  for (int r = 0; r < g; ++r) {
    w8 = max(w8, bands[2 * r]);
    w4 = max(w4, bands[2 * r + 1]);
  }
  HeadRuns h;
  h.keep = ex ? min(1, tiles) : max(1, tiles - max(w8, w4));
  h.k8 = max(1, tiles - w8);
  h.v8 = max(h.keep, tiles - NEAR_V8);
  return h;
}

__global__ __launch_bounds__(STORE_THREADS) void cache_store_kernel(CacheStoreArgs a) {
  __shared__ int sb[2 * STORE_MAX_HQ];
  __shared__ int4 sc[STORE_MAX_HQ];  // per KV head: INT4-K, INT8-K, INT8-V and INT4-V tiles
  const int tid = threadIdx.x;
  const int chunk = blockIdx.x, kh = blockIdx.y, s = blockIdx.z;
  const int g = a.hq / a.hk, tiles = a.tiles, row = a.row0 + s;
  for (int i = tid; i < 2 * a.hq; i += STORE_THREADS) sb[i] = a.bands[i];
  __syncthreads();
  for (int h = tid; h < a.hk; h += STORE_THREADS) {
    int4 c = make_int4(0, 0, 0, 0);
    if (a.exact == nullptr || a.exact[h] < 0) {
      const HeadRuns r = head_runs(sb + 2 * h * g, g, false, tiles);
      c = make_int4(r.k8 - r.keep, 1 + tiles - r.k8, 1 + tiles - r.v8, r.v8 - r.keep);
    }
    sc[h] = c;
  }
  __syncthreads();
  // record numbering is (KV head, entry) order within a sequence: the counts of the heads before kh, and the
  // sequence's totals
  int4 before = make_int4(0, 0, 0, 0), total = before;
  for (int h = 0; h < a.hk; ++h) {
    const int4 c = sc[h];
    if (h == kh) before = total;
    total = make_int4(total.x + c.x, total.y + c.y, total.z + c.z, total.w + c.w);
  }
  const bool ex = a.exact != nullptr && a.exact[kh] >= 0;
  const int xs = ex ? a.exact[kh] : 0;
  const HeadRuns runs = head_runs(sb + 2 * kh * g, g, ex, tiles);
  const int64_t base4 = a.o4 + (int64_t)s * total.x + before.x, base8 = a.o8 + (int64_t)s * total.y + before.y;
  const int64_t basev8 = a.ov8 + (int64_t)s * total.z + before.z, basev4 = a.ov4 + (int64_t)s * total.w + before.w;
  // K and V record slots of kept tile j of this (quantized) head
  auto is4 = [&](int j) { return !ex && j > 0 && j < runs.k8; };
  auto v8 = [&](int j) { return j == 0 || j >= runs.v8; };
  auto kslot = [&](int j) { return is4(j) ? base4 + (j - runs.keep) : base8 + (j == 0 ? 0 : 1 + (j - runs.k8)); };
  auto vslot = [&](int j) { return !v8(j) ? basev4 + (j - runs.keep) : basev8 + (j == 0 ? 0 : 1 + (j - runs.v8)); };
  const int64_t hb_src = (int64_t)s * a.hk + kh;
  const int64_t hb = (int64_t)row * a.hk + kh;
  // the chunk's kept records
  const int jend = min(tiles, (chunk + 1) * a.chunk);
  for (int j = chunk * a.chunk; j < jend; ++j) {
    if (j > 0 && j < runs.keep) continue;
    const uint8_t *ks, *vs;
    uint8_t *kd, *vd;
    int kbytes, vbytes;
    if (ex) {
      const int64_t src = ((int64_t)s * a.nx + xs) * tiles + j;
      const int64_t dst = a.ox + ((int64_t)s * a.nx + xs) * a.xstride + j;
      ks = a.kx + src * KX_BYTES;
      vs = a.vx + src * KX_BYTES;
      kd = a.kxc + dst * KX_BYTES;
      vd = a.vxc + dst * KX_BYTES;
      kbytes = vbytes = dst < a.capx ? KX_BYTES : 0;
    } else {
      const int64_t src = hb_src * tiles + j, kn = kslot(j), vn = vslot(j);
      const bool k4 = is4(j), v4 = !v8(j);
      ks = k4 ? a.k4p + src * K4_BYTES : a.kp + src * K8_BYTES;
      kd = k4 ? a.k4c + kn * K4_BYTES : a.k8c + kn * K8_BYTES;
      kbytes = k4 ? (kn < a.cap4 && a.k4p != nullptr ? K4_BYTES : 0) : (kn < a.cap8 ? K8_BYTES : 0);
      vs = v4 ? a.v4p + src * V4_BYTES : a.v8p + src * V8_BYTES;
      vd = v4 ? a.v4c + vn * V4_BYTES : a.v8c + vn * V8_BYTES;
      vbytes = v4 ? (vn < a.capv4 && a.v4p != nullptr ? V4_BYTES : 0) : (vn < a.capv8 ? V8_BYTES : 0);
    }
    constexpr int STEP = STORE_THREADS * 16, STEPS = KX_BYTES / STEP;
    v4i kw[STEPS], vw[STEPS];
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int off = i * STEP + tid * 16;
      if (off < kbytes) kw[i] = *reinterpret_cast<const v4i*>(ks + off);
      if (off < vbytes) vw[i] = *reinterpret_cast<const v4i*>(vs + off);
    }
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int off = i * STEP + tid * 16;
      if (off < kbytes) *reinterpret_cast<v4i*>(kd + off) = kw[i];
      if (off < vbytes) *reinterpret_cast<v4i*>(vd + off) = vw[i];
    }
  }
  if (chunk != 0 || row >= a.rows) return;
  // the head's metadata row
  const int cnt = 1 + tiles - runs.keep;
  for (int e = tid; e < a.maxn; e += STORE_THREADS) {
    int entry = 0, info = 0, slot = 0;
    if (e < cnt) {
      const int j = e == 0 ? 0 : runs.keep + e - 1, d = tiles - 1 - j;
      int mask = 0;
      for (int r = 0; r < g; ++r) {
        const bool on = ex || j == 0 || d < sb[2 * (kh * g + r)] || d < sb[2 * (kh * g + r) + 1];
        mask |= (on ? 1 : 0) << r;
      }
      entry = j | (1 << 30) | (j == 0 || d < NEAR_V8 ? 1 << 29 : 0);
      info = (mask & 0xff) | (is4(j) ? 1 << 8 : 0) | (int)((uint32_t)(ex ? 0 : kslot(j)) << 9);
      slot = ex ? 0 : (int)vslot(j);
    }
    a.entry[hb * a.maxn + e] = entry;
    a.kinfo[hb * a.maxn + e] = info;
    a.slot[hb * a.maxn + e] = slot;
  }
  if (tid == 0) {
    a.count[hb] = cnt;
    if (a.xslot) a.xslot[hb] = ex ? (int)(a.ox + ((int64_t)s * a.nx + xs) * a.xstride) : -1;
  }
  for (int i = tid; i < a.tiles_max * 4; i += STORE_THREADS) {
    a.ka_c[hb * a.tiles_max * 4 + i] = i < tiles * 4 ? a.ka[hb_src * tiles * 4 + i] : 1.f;
    if (a.ka4_c) a.ka4_c[hb * a.tiles_max * 4 + i] = (i < tiles * 4 && a.ka4) ? a.ka4[hb_src * tiles * 4 + i] : 1.f;
  }
  for (int i = tid; i < 3 * D; i += STORE_THREADS) {
    a.kstat_c[hb * 3 * D + i] = a.kstat[hb_src * 3 * D + i];
    a.vstat_c[hb * 3 * D + i] = a.vstat[hb_src * 3 * D + i];
  }
  if (kh == 0) {
    if (tid == 0) a.prompt[row] = a.t;
    for (int j = tid; j < a.tiles_max; j += STORE_THREADS)
      a.fmt[(int64_t)row * a.tiles_max + j] = (j < tiles && !(j == 0 || tiles - 1 - j < NEAR_V8)) ? 2 : 1;
  }
}

}  // namespace tri
