// Shared definitions of the SYCLDB operator library for MI355X (gfx950).
//
// The per-row integer semantics live in sdb_semantics.hpp.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <stdexcept>
#include <string>

#include "sdb_semantics.hpp"

namespace sdb {

// Error carrying a C-ABI status code; converted at the boundary.
struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

[[noreturn]] inline void fail(int code, const std::string &msg) { throw Error(code, msg); }

inline void hip_check(hipError_t e, const char *what)
{
    if (e != hipSuccess)
        fail(SDB_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

#define SDB_HIP(call) ::sdb::hip_check((call), #call)

// ------------------------------------------------------------- launch shape

// Number of compute units of the current device (cached per device).
int device_cu_count();
// Grid for a grid-stride streaming kernel over `units` work items with
// `per_block` items consumed per block iteration.
unsigned stream_grid(int64_t units, int64_t per_block, int blocks_per_cu = 8);

// Library-owned scratch: a device buffer of at least `bytes` for the calls of
// one stream.  Work of a stream runs in order, so a call's kernels are done
// with the buffer before the next call's overwrite it; calls on different
// streams get different buffers.  Held while the kernels that use it are
// queued, so that two threads on one stream do not mix theirs.  A call that is
// being captured gets a buffer of its stream's captures, which is never freed
// or moved: the graph keeps its address.  (Graphs captured on one stream share
// it: their replays must not overlap.)
struct ScratchBuffer;
class Scratch {
  public:
    Scratch(size_t bytes, hipStream_t stream);
    ~Scratch();
    Scratch(const Scratch &) = delete;
    Scratch &operator=(const Scratch &) = delete;
    uint8_t *data() const;

  private:
    std::shared_ptr<ScratchBuffer> buf_;
};
// Gives back the buffer of a stream about to be destroyed (its work done).
void scratch_release(hipStream_t stream);

// ------------------------------------------------------- result transfer

// Ids of the rows whose flag is set, in row order, into row_ids (capacity n);
// their number into *count.  tile_counts: compact_tiles(n) words of device
// memory for the per-tile counts.
int64_t compact_tiles(int64_t n);
void launch_compact_into(const uint8_t *flags, int64_t n, int32_t *row_ids, uint32_t *count, uint32_t *tile_counts,
                         hipStream_t s);
// dst[c][j] = src[c][ids[j]] for j < count (0 where ids[j] >= src_rows[c]);
// a column holds int32 values, or uint64 where bit c of is_u64 is set.
constexpr int GATHER_MAX_COLS = 8;
struct GatherCols {
    const void *src[GATHER_MAX_COLS];
    void *dst[GATHER_MAX_COLS];
    uint64_t src_rows[GATHER_MAX_COLS];
    uint32_t is_u64;
    int32_t ncols;
};
void launch_gather_cols(const GatherCols &g, const int32_t *ids, int64_t count, hipStream_t s);
// Writes bytes[i] bytes to dst + off[i] for every part: several small arrays
// packed into one buffer, in device memory or in pinned host memory.
enum PackKind : uint8_t {
    PACK_COPY = 0, // the bytes at src[i]
    PACK_SEEN = 1, // flags: 1 where the uint32 at src[i] is nonzero
    PACK_TRUE = 2  // flags: all 1 (no source)
};
constexpr int PACK_MAX_PARTS = 64;
struct PackParts {
    const uint8_t *src[PACK_MAX_PARTS];
    uint64_t off[PACK_MAX_PARTS];
    uint64_t bytes[PACK_MAX_PARTS];
    uint8_t kind[PACK_MAX_PARTS];
    int32_t n;
};
void launch_pack_parts(const PackParts &p, uint8_t *dst, hipStream_t s);

// The selected rows of tables of up to SPARSE_MAX_ROWS rows, in row order:
// their ids, their values of every column (as launch_gather_cols) and their
// number, written to dst / ids / count (pinned host memory).  A row is
// selected where its flag (or, without flags, its `seen` word) is nonzero.
// counts: sparse_tiles(rows) words of device memory.
constexpr uint64_t SPARSE_MAX_ROWS = 1u << 22;
struct SparseTable {
    const uint8_t *flags;
    const uint32_t *seen;
    uint32_t *counts;
    const void *src[GATHER_MAX_COLS];
    void *dst[GATHER_MAX_COLS];
    uint32_t src_rows[GATHER_MAX_COLS];
    uint32_t *ids, *count;
    uint32_t rows, is_u64;
    int32_t ncols;
};
uint64_t sparse_tiles(uint64_t rows);
int launch_sparse_tables(const SparseTable *t, size_t n, hipStream_t s); // number of launches

// Statistics of compact probe tables, each stats[i] laid out as [overflow
// flag, nparts[i] partial counts]: the sums and flags go to dst as pairs.
struct StatsParts {
    const uint32_t *stats[PACK_MAX_PARTS];
    uint32_t nparts[PACK_MAX_PARTS];
    int32_t n;
};
void launch_stats_reduce(const StatsParts &p, uint32_t *dst, hipStream_t s);

// One compact table to build.  dict (or null): the rank dictionary
// (FV_RANK16 layout, capacity dict_cap bytes) of its presence bitmap and
// 16-bit values is built too.
struct CompactJob {
    const void *ht;
    bool pairs;          // (flag, value) pairs, else uint8 keys
    int32_t len, vmin;
    uint32_t *bits;
    uint16_t *vals;      // 16-bit value offsets, or null
    uint32_t *partials, *bad;
    uint8_t *dict;
    uint32_t dict_cap;
};
// Builds them in one launch per COMPACT_JOBS tables (two with dictionaries);
// returns the number of launches.
int launch_compact_tables(const CompactJob *jobs, size_t njobs, hipStream_t s);

} // namespace sdb
