// Tables of the intra-stage search to host arrays, strategy rows decoded on the way.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <utility>

#include "mist_common.h"
#include "mist_search.h"

using mist::fail;

namespace {

// A chunk of output in pinned memory, made of pieces of the caller's arrays.
constexpr int kFetchPieces = 16;
constexpr size_t kFetchChunk = (size_t)1 << 20;
constexpr int kFetchSlots = 3;
constexpr int kFetchBlocks = 128;
constexpr int kRowFields = 10;
struct FetchPiece {
  const void *from;
  int64_t to;       // byte in the chunk, a multiple of 16
  int64_t count;    // doubles, or indices
  int32_t rows, group;
};
struct FetchPieces {
  FetchPiece piece[kFetchPieces];
  int32_t n;
};

// (b, dp, tp, wre, gre, ore, wo, go, oo, ao) of a row, reference order (batched_module_analyzer.py:490-534): field
// pair `k` of it; a cell without a row holds +inf.
__device__ __forceinline__ double2 row_fields(const MistGroupDesc *__restrict__ g, int32_t index, int k) {
  if (index < 0 || g == nullptr || index >= g->n_rows) return make_double2(INFINITY, INFINITY);
  const uint32_t n_ao = (uint32_t)g->n_ao, n_tail = (uint32_t)g->n_oo * n_ao, n_off = (uint32_t)g->n_off;
  const uint32_t par = (uint32_t)index / n_off, off = (uint32_t)index - par * n_off;
  if (k < 3) return make_double2(g->par[par][2 * k], g->par[par][2 * k + 1]);
  const uint32_t pair = off / n_tail, tail = off - pair * n_tail;
  if (k == 3) return make_double2(g->wo[g->pair_wo[pair]], g->go[g->pair_go[pair]]);
  return make_double2(g->oo[tail / n_ao], g->ao[tail % n_ao]);
}
static_assert(MIST_PAR_B == 0 && MIST_PAR_ORE == 5, "the first six fields of a row");

// Written straight into pinned host memory, in whole lines.  Bound: the link to the host, 50 GB/s, and the copy out of
// the chunks beside it: 68700 cells of 7B on 2x8, 6.6 MB, 0.16 ms with the calls.  (Twelve copies to pageable memory,
// 17 GB/s, and the rows decoded there by numpy, 0.75 ms of divisions and gathers: 1.1 ms.  The decoded rows through
// one such copy would take 0.39.)
__global__ __launch_bounds__(256) void fetch_kernel(const FetchPieces pieces, const MistGroupDesc *__restrict__ groups,
                                                    char *__restrict__ chunk) {
  const int64_t me = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, all = (int64_t)gridDim.x * blockDim.x;
  for (int i = 0; i < pieces.n; ++i) {
    const FetchPiece &piece = pieces.piece[i];
    if (piece.rows == 0) {
      const double *__restrict__ from = static_cast<const double *>(piece.from);
      double *to = reinterpret_cast<double *>(chunk + piece.to);
      for (int64_t e = me; e < piece.count; e += all) to[e] = from[e];
    } else {
      const int32_t *__restrict__ from = static_cast<const int32_t *>(piece.from);
      double2 *to = reinterpret_cast<double2 *>(chunk + piece.to);
      const MistGroupDesc *g = piece.group < 0 ? nullptr : groups + piece.group;
      constexpr int kPairs = kRowFields / 2;
      for (int64_t e = me; e < piece.count * kPairs; e += all) to[e] = row_fields(g, from[e / kPairs], (int)(e % kPairs));
    }
  }
}

// Pinned chunks and their events, kFetchSlots MB.  A fetch has a ring to itself, so that those of several threads
// and devices wait for nothing of each other.  The last kFetchKept rings are kept for the next fetches, for the life
// of the process; a fetch that finds none of its device makes one.
constexpr int kFetchKept = 8;
struct FetchRing {
  int device;
  char *chunk[kFetchSlots];
  hipEvent_t filled[kFetchSlots];
};
std::mutex g_fetch_lock;  // of the kept rings, not held while anything is waited for
FetchRing g_fetch_rings[kFetchKept];
int g_fetch_n_kept = 0, g_fetch_oldest = 0;

void free_ring(const FetchRing &ring) {
  for (int i = 0; i < kFetchSlots; ++i) {
    if (ring.chunk[i] != nullptr) (void)hipHostFree(ring.chunk[i]);
    if (ring.filled[i] != nullptr) (void)hipEventDestroy(ring.filled[i]);
  }
}

int take_ring(FetchRing *ring) {
  MIST_HIP_CHECK(hipGetDevice(&ring->device));
  {
    std::lock_guard<std::mutex> guard(g_fetch_lock);
    for (int i = 0; i < g_fetch_n_kept; ++i)
      if (g_fetch_rings[i].device == ring->device) {
        *ring = g_fetch_rings[i];
        g_fetch_rings[i] = g_fetch_rings[--g_fetch_n_kept];
        return 0;
      }
  }
  for (int i = 0; i < kFetchSlots; ++i) {
    MIST_HIP_CHECK(hipHostMalloc(reinterpret_cast<void **>(&ring->chunk[i]), kFetchChunk, hipHostMallocCoherent));
    MIST_HIP_CHECK(hipEventCreateWithFlags(&ring->filled[i], hipEventDisableTiming));
  }
  return 0;
}

// (of a ring that nothing writes to any more)
void give_back_ring(FetchRing ring) {
  {
    std::lock_guard<std::mutex> guard(g_fetch_lock);
    if (g_fetch_n_kept < kFetchKept) {
      g_fetch_rings[g_fetch_n_kept++] = ring;
      return;
    }
    std::swap(ring, g_fetch_rings[g_fetch_oldest]);  // (which may be one of another device)
    g_fetch_oldest = (g_fetch_oldest + 1) % kFetchKept;
  }
  free_ring(ring);
}

// Chunk by chunk: the next ones are written while one is copied out to the caller's arrays.
int fetch_items(const MistFetchItem *items, int n_items, const MistGroupDesc *d_groups, const FetchRing &ring, hipStream_t stream) {
  struct Part {  // of a chunk: where a piece goes
    char *to;
    int64_t at, bytes;
  };
  Part parts[kFetchSlots][kFetchPieces];
  int n_parts[kFetchSlots] = {};
  int item = 0;
  int64_t done = 0;  // elements of the item
  auto fill = [&](int slot) -> int {
    FetchPieces pieces = {};
    int64_t used = 0;
    while (item < n_items && pieces.n < kFetchPieces) {
      const MistFetchItem &it = items[item];
      const int64_t each = it.rows ? kRowFields * (int64_t)sizeof(double) : (int64_t)sizeof(double);
      const int64_t count = std::min(it.count - done, ((int64_t)kFetchChunk - used) / each);
      if (count <= 0 && done < it.count) break;  // the chunk is full
      if (count > 0) {
        const int k = pieces.n++;
        const char *from = static_cast<const char *>(it.from) + done * (it.rows ? (int64_t)sizeof(int32_t) : each);
        pieces.piece[k] = FetchPiece{from, used, count, it.rows, it.group};
        parts[slot][k] = Part{static_cast<char *>(it.to) + done * each, used, count * each};
        used = (used + count * each + 15) / 16 * 16;
        done += count;
      }
      if (done == it.count) {
        ++item;
        done = 0;
      }
    }
    n_parts[slot] = pieces.n;
    if (pieces.n == 0) return 0;
    hipLaunchKernelGGL(fetch_kernel, dim3(kFetchBlocks), dim3(256), 0, stream, pieces, d_groups, ring.chunk[slot]);
    MIST_HIP_CHECK(hipGetLastError());
    MIST_HIP_CHECK(hipEventRecord(ring.filled[slot], stream));
    return 0;
  };
  for (int slot = 0; slot < kFetchSlots; ++slot)
    if (int rc = fill(slot)) return rc;
  for (int slot = 0; n_parts[slot] > 0; slot = (slot + 1) % kFetchSlots) {
    MIST_HIP_CHECK(hipEventSynchronize(ring.filled[slot]));
    for (int k = 0; k < n_parts[slot]; ++k)
      std::memcpy(parts[slot][k].to, ring.chunk[slot] + parts[slot][k].at, (size_t)parts[slot][k].bytes);
    if (int rc = fill(slot)) return rc;
  }
  return 0;
}

}  // namespace

extern "C" {

int mist_sizeof_fetch_item(void) { return (int)sizeof(MistFetchItem); }

int mist_fetch_tables(const MistFetchItem *items, int n_items, const MistGroupDesc *d_groups, int n_groups, void *stream) {
  if (!items || n_items < 1) return fail(MIST_E_INVALID, "nothing to fetch");
  for (int i = 0; i < n_items; ++i) {
    if (!items[i].from || !items[i].to || items[i].count < 0)
      return fail(MIST_E_INVALID, "item %d: null pointer or %lld elements", i, (long long)items[i].count);
    if (items[i].rows && (items[i].group >= n_groups || (items[i].group >= 0 && !d_groups)))
      return fail(MIST_E_INVALID, "item %d: group %d of %d", i, items[i].group, n_groups);
  }
  FetchRing ring = {};
  int rc = take_ring(&ring);
  if (rc == 0) rc = fetch_items(items, n_items, d_groups, ring, (hipStream_t)stream);
  if (rc != 0) {
    (void)hipStreamSynchronize((hipStream_t)stream);  // (the chunks may still be written)
    free_ring(ring);
    return rc;
  }
  give_back_ring(ring);
  return 0;
}

}  // extern "C"
