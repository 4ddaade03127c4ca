// Operator kernels of the drop-in per-operator path (one launch per
// reference functor) and their C-ABI entry points.
//
// Layout: int32 columns and 1-byte flags in HBM.  A thread handles chunks of
// 4 consecutive rows (one 16-byte column load, one 32-bit flag word), a block
// handles 256 x UNROLL chunks per step, the grid strides over the column.  All
// loads of a step are issued before any store so each wave keeps UNROLL
// vector loads in flight.  Comparison / logic / arithmetic variants are
// template parameters so the row loop carries no data-independent branches.
// Pointers that are not 16-byte (columns) or 4-byte (flags) aligned take a
// one-row-per-thread path instead.
#include "capi_util.hpp"
#include "fused_types.hpp"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

namespace sdb {
namespace {

constexpr int BLOCK = 256;
constexpr int UNROLL = 4;
constexpr uint32_t LDS_PER_CU = 160 * 1024; // gfx950
constexpr int64_t ROWS_PER_STEP = (int64_t)BLOCK * UNROLL * 4;

inline bool aligned(const void *p, size_t a) { return ((uintptr_t)p % a) == 0; }

__device__ __forceinline__ uint32_t byte_of(uint32_t w, int k) { return (w >> (8 * k)) & 0xffu; }

// ------------------------------------------------------------- selection

template <int CMP, int LOGIC>
__global__ void __launch_bounds__(BLOCK) k_select_lit(const int32_t *__restrict__ col,
                                                      const uint8_t *in, uint8_t *out, int64_t n,
                                                      int32_t v)
{
    const int64_t nchunks = n >> 2;
    const int4 *c4 = reinterpret_cast<const int4 *>(col);
    const uint32_t *in32 = reinterpret_cast<const uint32_t *>(in);
    uint32_t *out32 = reinterpret_cast<uint32_t *>(out);
    for (int64_t base = (int64_t)blockIdx.x * BLOCK * UNROLL; base < nchunks;
         base += (int64_t)gridDim.x * BLOCK * UNROLL) {
        int4 x[UNROLL];
        uint32_t f[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            const int64_t c = base + u * BLOCK + threadIdx.x;
            if (c < nchunks) {
                x[u] = c4[c];
                f[u] = (LOGIC == SDB_NONE) ? 0u : in32[c];
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            const int64_t c = base + u * BLOCK + threadIdx.x;
            if (c < nchunks) {
                const int32_t xs[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
                uint32_t r = 0;
#pragma unroll
                for (int k = 0; k < 4; k++)
                    r |= (uint32_t)logical(LOGIC, byte_of(f[u], k) != 0, compare(CMP, xs[k], v)) << (8 * k);
                out32[c] = r;
            }
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {
        const int64_t i = (nchunks << 2) + threadIdx.x;
        out[i] = logical(LOGIC, in[i] != 0, compare(CMP, col[i], v));
    }
}

template <int CMP, int LOGIC>
__global__ void __launch_bounds__(BLOCK) k_select_lit_row(const int32_t *col, const uint8_t *in,
                                                          uint8_t *out, int64_t n, int32_t v)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK)
        out[i] = logical(LOGIC, in[i] != 0, compare(CMP, col[i], v));
}

template <int CMP, int LOGIC>
__global__ void __launch_bounds__(BLOCK) k_select_col(const int32_t *__restrict__ a,
                                                      const int32_t *__restrict__ b,
                                                      const uint8_t *in, uint8_t *out, int64_t n)
{
    const int64_t nchunks = n >> 2;
    const int4 *a4 = reinterpret_cast<const int4 *>(a);
    const int4 *b4 = reinterpret_cast<const int4 *>(b);
    const uint32_t *in32 = reinterpret_cast<const uint32_t *>(in);
    uint32_t *out32 = reinterpret_cast<uint32_t *>(out);
    for (int64_t base = (int64_t)blockIdx.x * BLOCK * UNROLL; base < nchunks;
         base += (int64_t)gridDim.x * BLOCK * UNROLL) {
        int4 x[UNROLL], y[UNROLL];
        uint32_t f[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            const int64_t c = base + u * BLOCK + threadIdx.x;
            if (c < nchunks) {
                x[u] = a4[c];
                y[u] = b4[c];
                f[u] = (LOGIC == SDB_NONE) ? 0u : in32[c];
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            const int64_t c = base + u * BLOCK + threadIdx.x;
            if (c < nchunks) {
                const int32_t xs[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
                const int32_t ys[4] = {y[u].x, y[u].y, y[u].z, y[u].w};
                uint32_t r = 0;
#pragma unroll
                for (int k = 0; k < 4; k++)
                    r |= (uint32_t)logical(LOGIC, byte_of(f[u], k) != 0, compare(CMP, xs[k], ys[k])) << (8 * k);
                out32[c] = r;
            }
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {
        const int64_t i = (nchunks << 2) + threadIdx.x;
        out[i] = logical(LOGIC, in[i] != 0, compare(CMP, a[i], b[i]));
    }
}

template <int CMP, int LOGIC>
__global__ void __launch_bounds__(BLOCK) k_select_col_row(const int32_t *a, const int32_t *b,
                                                          const uint8_t *in, uint8_t *out, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK)
        out[i] = logical(LOGIC, in[i] != 0, compare(CMP, a[i], b[i]));
}

template <int LOGIC>
__global__ void __launch_bounds__(BLOCK) k_logical(const uint8_t *in, const uint8_t *local,
                                                   uint8_t *out, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK)
        out[i] = logical(LOGIC, in[i] != 0, local[i] != 0);
}

// 0x01 in each byte of x that is nonzero, 0x00 elsewhere (no carry crosses a
// byte: (b & 0x7f) + 0x7f <= 0xfe)
__device__ __forceinline__ uint32_t nz_bytes(uint32_t x)
{
    return ((((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) >> 7) & 0x01010101u;
}

template <int LOGIC> __device__ __forceinline__ uint32_t logical_bytes(uint32_t a, uint32_t b)
{
    return LOGIC == SDB_NONE ? nz_bytes(b) : LOGIC == SDB_AND ? (nz_bytes(a) & nz_bytes(b)) : (nz_bytes(a) | nz_bytes(b));
}

// The same, 16 flags per thread and step (the three buffers 16-byte
// aligned); the last n % 16 flags one per thread.
template <int LOGIC>
__global__ void __launch_bounds__(BLOCK) k_logical_vec(const uint8_t *in, const uint8_t *local, uint8_t *out,
                                                       int64_t n)
{
    const int64_t nq = n >> 4;
    const uint4 *a4 = reinterpret_cast<const uint4 *>(in);
    const uint4 *b4 = reinterpret_cast<const uint4 *>(local);
    uint4 *o4 = reinterpret_cast<uint4 *>(out);
    for (int64_t base = (int64_t)blockIdx.x * BLOCK * UNROLL; base < nq; base += (int64_t)gridDim.x * BLOCK * UNROLL) {
        uint4 a[UNROLL], b[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            const int64_t c = base + u * BLOCK + threadIdx.x;
            if (c < nq) {
                a[u] = LOGIC == SDB_NONE ? make_uint4(0, 0, 0, 0) : a4[c];
                b[u] = b4[c];
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            const int64_t c = base + u * BLOCK + threadIdx.x;
            if (c < nq)
                o4[c] = make_uint4(logical_bytes<LOGIC>(a[u].x, b[u].x), logical_bytes<LOGIC>(a[u].y, b[u].y),
                                   logical_bytes<LOGIC>(a[u].z, b[u].z), logical_bytes<LOGIC>(a[u].w, b[u].w));
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 15)) {
        const int64_t i = (nq << 4) + threadIdx.x;
        out[i] = logical(LOGIC, in[i] != 0, local[i] != 0);
    }
}

// ------------------------------------------------------------ projection

__global__ void __launch_bounds__(BLOCK) k_fill_i32(int32_t *dst, int32_t v, int64_t n)
{
    const int64_t head = ((16 - ((uintptr_t)dst & 15)) & 15) / 4; // rows before 16B boundary
    const int64_t h = head < n ? head : n;
    if (blockIdx.x == 0 && threadIdx.x < h) dst[threadIdx.x] = v;
    int32_t *body = dst + h;
    const int64_t m = n - h;
    const int64_t nchunks = m >> 2;
    int4 *d4 = reinterpret_cast<int4 *>(body);
    const int4 vv = make_int4(v, v, v, v);
    for (int64_t c = (int64_t)blockIdx.x * BLOCK + threadIdx.x; c < nchunks; c += (int64_t)gridDim.x * BLOCK)
        d4[c] = vv;
    if (blockIdx.x == 0 && threadIdx.x < (m & 3)) body[(nchunks << 2) + threadIdx.x] = v;
}

// 16-byte stores between the first and the last 16-byte boundary of the
// buffer; the head and tail bytes (fewer than 16 each) one per thread
__global__ void __launch_bounds__(BLOCK) k_fill_u8(uint8_t *dst, uint8_t v, int64_t n)
{
    const int64_t head = min(n, (int64_t)((16u - ((uintptr_t)dst & 15u)) & 15u));
    const int64_t nq = (n - head) >> 4, tail0 = head + (nq << 4);
    const uint32_t w = 0x01010101u * v;
    const uint4 q = make_uint4(w, w, w, w);
    uint4 *dq = reinterpret_cast<uint4 *>(dst + head);
    const int64_t tid = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    for (int64_t i = tid; i < nq; i += (int64_t)gridDim.x * BLOCK) dq[i] = q;
    if (tid < head) dst[tid] = v;
    if (tid < n - tail0) dst[tail0 + tid] = v;
}

__global__ void k_zero_u64(uint64_t *p) { *p = 0; }

// kind: 0 = column op column, 1 = literal op column, 2 = column op literal
template <int OP, int KIND>
__global__ void __launch_bounds__(BLOCK) k_binop(int32_t *result, const int32_t *a, const int32_t *b,
                                                 int32_t lit, const uint8_t *flags, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK) {
        if (flags[i]) {
            const int32_t x = KIND == 1 ? lit : a[i];
            const int32_t y = KIND == 2 ? lit : b[i];
            result[i] = element_op(OP, x, y);
        }
    }
}

// Vector form: 4 rows per chunk, rows whose flag is 0 keep their content.
template <int OP, int KIND>
__global__ void __launch_bounds__(BLOCK) k_binop_vec(int32_t *result, const int32_t *a,
                                                     const int32_t *b, int32_t lit,
                                                     const uint8_t *flags, int64_t n)
{
    const int64_t nchunks = n >> 2;
    const uint32_t *f32 = reinterpret_cast<const uint32_t *>(flags);
    for (int64_t base = (int64_t)blockIdx.x * BLOCK * UNROLL; base < nchunks;
         base += (int64_t)gridDim.x * BLOCK * UNROLL) {
        uint32_t f[UNROLL];
        int4 x[UNROLL], y[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            const int64_t c = base + u * BLOCK + threadIdx.x;
            f[u] = c < nchunks ? f32[c] : 0u;
            if (f[u]) {
                if (KIND != 1) x[u] = reinterpret_cast<const int4 *>(a)[c];
                if (KIND != 2) y[u] = reinterpret_cast<const int4 *>(b)[c];
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            if (!f[u]) continue;
            const int64_t c = base + u * BLOCK + threadIdx.x;
            const int32_t xs[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
            const int32_t ys[4] = {y[u].x, y[u].y, y[u].z, y[u].w};
            int32_t r[4];
#pragma unroll
            for (int k = 0; k < 4; k++)
                r[k] = element_op(OP, KIND == 1 ? lit : xs[k], KIND == 2 ? lit : ys[k]);
            if (f[u] == 0x01010101u) {
                reinterpret_cast<int4 *>(result)[c] = make_int4(r[0], r[1], r[2], r[3]);
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (byte_of(f[u], k)) result[4 * c + k] = r[k];
            }
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {
        const int64_t i = (nchunks << 2) + threadIdx.x;
        if (flags[i]) result[i] = element_op(OP, KIND == 1 ? lit : a[i], KIND == 2 ? lit : b[i]);
    }
}

// ------------------------------------------------------- tiles of a wave

// Tiles of WT_ROWS rows per wave: chunk j of a lane holds the rows
// t0 + 256 j + 4 lane .. + 3, so that flags (4 bytes) and columns (16 bytes)
// load coalesced; bit 4 j + k of a lane's 32-bit row mask is row k of its
// chunk j.
constexpr int WT_CHUNKS = 8;
constexpr int64_t WT_ROWS = 256 * WT_CHUNKS;

__device__ __forceinline__ int64_t wt_row(int64_t t0, int lane, int j) { return t0 + 256 * j + 4 * lane; }
// offset in its tile of the row of mask bit b
__device__ __forceinline__ uint32_t wt_offset(int lane, uint32_t b) { return (b >> 2) * 256u + 4u * lane + (b & 3u); }

// Flags of a whole tile, at any alignment (global memory takes wide loads at
// any byte).  The rows past the last whole tile are left to the last block's
// threads, one each: read here with bounds checks they cost a round trip per
// row slot, and the registers that a second block per CU needs.
__device__ __forceinline__ void wt_flags(const uint8_t *flags, int64_t t0, int lane, uint32_t (&f)[WT_CHUNKS])
{
#pragma unroll
    for (int j = 0; j < WT_CHUNKS; j++) __builtin_memcpy(&f[j], flags + wt_row(t0, lane, j), 4);
}

// Bit k: whether byte k of x is nonzero (the flag bits 0, 8, 16, 24 of
// nz_bytes meet in bits 24..27 of the product, with no carry into them).
__device__ __forceinline__ uint32_t nz_mask(uint32_t x) { return (nz_bytes(x) * 0x01020408u) >> 24; }

// The flags 0 / 1 of the low four bits of m, one per byte
__device__ __forceinline__ uint32_t flag_bytes(uint32_t m) { return ((m & 15u) * 0x00204081u) & 0x01010101u; }

__device__ __forceinline__ uint32_t wt_mask(const uint32_t (&f)[WT_CHUNKS])
{
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < WT_CHUNKS; j++) m |= nz_mask(f[j]) << (4 * j);
    return m;
}

// The wave's index in its block, in a scalar register: addresses that follow
// from it (a tile's) then are scalar bases with 32-bit offsets per lane.
__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// LDS written by some lanes of a wave and read by others
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Exclusive prefix of v over the lanes of the wave, and the total.
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v, int lane, uint32_t &total)
{
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    total = __builtin_amdgcn_readlane(x, 63);
    return x - v;
}

// Block-wide min and max (BLOCK threads), valid in thread 0
__device__ __forceinline__ void block_minmax(int32_t &lo, int32_t &hi)
{
    for (int off = 32; off > 0; off >>= 1) {
        lo = min(lo, __shfl_xor(lo, off, 64));
        hi = max(hi, __shfl_xor(hi, off, 64));
    }
    __shared__ int32_t wlo[BLOCK / 64], whi[BLOCK / 64];
    if ((threadIdx.x & 63) == 0) {
        wlo[threadIdx.x >> 6] = lo;
        whi[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    for (int w = 0; w < BLOCK / 64; w++) {
        lo = min(lo, wlo[w]);
        hi = max(hi, whi[w]);
    }
}

// ------------------------------------------------------------------ join

__global__ void __launch_bounds__(BLOCK) k_build_keys(const int32_t *keys, const uint8_t *flags,
                                                      int64_t n, uint8_t *ht, int32_t len,
                                                      int32_t min)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK) {
        const uint32_t s = slot_of(keys[i], min);
        if (s < (uint32_t)len) ht[s] = flags[i] ? 1 : 0;
    }
}

__global__ void __launch_bounds__(BLOCK) k_build_keyvals(const int32_t *keys, const int32_t *vals,
                                                         const uint8_t *flags, int64_t n,
                                                         int32_t *ht, int32_t len, int32_t min)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK) {
        const uint32_t s = slot_of(keys[i], min);
        if (s >= (uint32_t)len) continue;
        if (flags[i])
            reinterpret_cast<int2 *>(ht)[s] = make_int2(1, vals[i]);
        else
            ht[2 * (int64_t)s] = 0;
    }
}

// vec: 4 rows per thread and step (keys 16-byte, flags 4-byte aligned),
// else one row.  The keys load beside the flags, not after them: one wait
// fewer per step, for the keys of chunks without a flagged row.
__global__ void __launch_bounds__(BLOCK) k_probe_semi(const int32_t *__restrict__ probe,
                                                      const uint8_t *in, uint8_t *out, int64_t n,
                                                      const uint8_t *__restrict__ ht, int32_t min,
                                                      int32_t max, int vec)
{
    auto present = [&](int32_t x) { return x >= min && x <= max && ht[slot_of(x, min)] != 0; };
    if (vec) {
        const int64_t nchunks = n >> 2;
        const int4 *p4 = reinterpret_cast<const int4 *>(probe);
        const uint32_t *in32 = reinterpret_cast<const uint32_t *>(in);
        uint32_t *out32 = reinterpret_cast<uint32_t *>(out);
        for (int64_t base = (int64_t)blockIdx.x * BLOCK * UNROLL; base < nchunks;
             base += (int64_t)gridDim.x * BLOCK * UNROLL) {
            uint32_t f[UNROLL];
            int4 x[UNROLL];
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                const int64_t c = base + u * BLOCK + threadIdx.x;
                f[u] = c < nchunks ? in32[c] : 0u;
                x[u] = c < nchunks ? p4[c] : make_int4(0, 0, 0, 0);
            }
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                const int64_t c = base + u * BLOCK + threadIdx.x;
                if (c >= nchunks) continue;
                uint32_t r = 0;
                if (f[u]) {
                    const int32_t xs[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const bool hit = byte_of(f[u], k) && present(xs[k]);
                        r |= (uint32_t)hit << (8 * k);
                    }
                }
                out32[c] = r;
            }
        }
        if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {
            const int64_t i = (nchunks << 2) + threadIdx.x;
            out[i] = in[i] && present(probe[i]);
        }
        return;
    }
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK) {
        const bool f = in[i] != 0;
        bool r = false;
        if (f) r = present(probe[i]);
        out[i] = r;
    }
}

// The semi probe of a long column.  The kernel above waits for each flagged
// row's table byte in turn, up to 16 round trips to L2 per step of a thread.
// Here a block first turns the table into a bitmap in LDS, one bit per slot,
// and the 16 answers of a step are read without a branch; two 1024-thread
// blocks per CU.  200M rows (the column and the flags alone take 228 us, what
// select_lit measures): 20,000 slots, every row flagged 381 -> 234 us, one in
// five 288 -> 235; 300,000 slots 345 -> 243; 61,130 slots, 5 % flagged 277 -> 236.
constexpr int SEMI_BLOCK = 1024;

__global__ void __launch_bounds__(SEMI_BLOCK) k_probe_semi_lds(const int32_t *__restrict__ probe, const uint8_t *in,
                                                               uint8_t *out, int64_t n, const uint8_t *__restrict__ ht,
                                                               uint32_t slots, int32_t min)
{
    extern __shared__ uint4 semi_lds[];
    uint16_t *const half = reinterpret_cast<uint16_t *>(semi_lds);
    for (uint32_t h = threadIdx.x; h < (slots + 15u) / 16u; h += SEMI_BLOCK) {
        uint32_t w[4] = {0, 0, 0, 0};
        if (16u * h + 16u <= slots) {
            const uint4 q = reinterpret_cast<const uint4 *>(ht)[h];
            w[0] = q.x;
            w[1] = q.y;
            w[2] = q.z;
            w[3] = q.w;
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 16u; k++)
                if (16u * h + k < slots) w[k >> 2] |= (uint32_t)ht[16u * h + k] << (8u * (k & 3u));
        }
        half[h] = (uint16_t)(nz_mask(w[0]) | nz_mask(w[1]) << 4 | nz_mask(w[2]) << 8 | nz_mask(w[3]) << 12);
    }
    __syncthreads();
    const uint32_t *const bits = reinterpret_cast<const uint32_t *>(semi_lds);
    const uint32_t last = (slots - 1u) >> 5;
    const int64_t nchunks = n >> 2;
    const int4 *p4 = reinterpret_cast<const int4 *>(probe);
    const uint32_t *in32 = reinterpret_cast<const uint32_t *>(in);
    uint32_t *out32 = reinterpret_cast<uint32_t *>(out);
    for (int64_t base = (int64_t)blockIdx.x * SEMI_BLOCK * UNROLL; base < nchunks;
         base += (int64_t)gridDim.x * SEMI_BLOCK * UNROLL) {
        uint32_t f[UNROLL];
        int4 x[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            const int64_t c = base + u * SEMI_BLOCK + threadIdx.x;
            f[u] = c < nchunks ? in32[c] : 0u;
            x[u] = c < nchunks ? p4[c] : make_int4(0, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            const int64_t c = base + u * SEMI_BLOCK + threadIdx.x;
            const int32_t xs[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
            uint32_t hit = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t s = (uint32_t)xs[k] - (uint32_t)min;
                const uint32_t w = bits[::min(s >> 5, last)]; // past the table: any word
                hit |= (uint32_t)(s < slots && ((w >> (s & 31u)) & 1u)) << k;
            }
            if (c < nchunks) out32[c] = flag_bytes(hit & nz_mask(f[u]));
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {
        const int64_t i = (nchunks << 2) + threadIdx.x;
        const uint32_t s = (uint32_t)probe[i] - (uint32_t)min;
        out[i] = in[i] && s < slots && ht[s] != 0;
    }
}

// The value table of a probe: the reference's (flag, value) pairs, or --
// when the caller's table is much smaller than the probe column -- a 16-bit
// copy built on the device just before (k_pairs_range, k_pairs_to_u16): one
// uint16 per slot, value - vmin where the flag is 1, VALS_UNSET elsewhere.
// A quarter of the bytes per gather keeps a table of millions of slots in
// L2; the device decides (info[2]) whether every value fitted, so the host
// never waits for it.
struct PairsOrU16 {
    const int2 *pairs;
    const uint16_t *u16; // null: pairs only
    const int32_t *info; // vmin, vmax, values do not fit in 16 bits
};

__device__ __forceinline__ bool probe_value(const PairsOrU16 &t, bool use16, int32_t vmin, uint32_t slot, int32_t &v)
{
    if (use16) {
        const uint32_t x = t.u16[slot];
        v = vmin + (int32_t)x;
        return x != VALS_UNSET;
    }
    const int2 e = t.pairs[slot];
    v = e.y;
    return e.x == 1;
}

__global__ void __launch_bounds__(BLOCK) k_probe_full(const int32_t *__restrict__ probe,
                                                      int32_t *val_out, const uint8_t *in,
                                                      uint8_t *out, int64_t n,
                                                      PairsOrU16 t, int32_t min,
                                                      int32_t max, int vec)
{
    const bool use16 = t.u16 && t.info[2] == 0;
    const int32_t vmin = t.u16 ? t.info[0] : 0;
    if (vec) {
        const int64_t nchunks = n >> 2;
        const int4 *p4 = reinterpret_cast<const int4 *>(probe);
        const uint32_t *in32 = reinterpret_cast<const uint32_t *>(in);
        uint32_t *out32 = reinterpret_cast<uint32_t *>(out);
        for (int64_t base = (int64_t)blockIdx.x * BLOCK * UNROLL; base < nchunks;
             base += (int64_t)gridDim.x * BLOCK * UNROLL) {
            uint32_t f[UNROLL];
            int4 x[UNROLL];
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                const int64_t c = base + u * BLOCK + threadIdx.x;
                f[u] = c < nchunks ? in32[c] : 0u;
                if (f[u]) x[u] = p4[c];
            }
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                const int64_t c = base + u * BLOCK + threadIdx.x;
                if (c >= nchunks) continue;
                uint32_t r = 0;
                if (f[u]) {
                    const int32_t xs[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        int32_t v;
                        if (byte_of(f[u], k) && xs[k] >= min && xs[k] <= max &&
                            probe_value(t, use16, vmin, slot_of(xs[k], min), v)) {
                            val_out[4 * c + k] = v;
                            r |= 1u << (8 * k);
                        }
                    }
                }
                out32[c] = r;
            }
        }
        if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {
            const int64_t i = (nchunks << 2) + threadIdx.x;
            bool r = false;
            if (in[i]) {
                const int32_t x = probe[i];
                int32_t v;
                if (x >= min && x <= max && probe_value(t, use16, vmin, slot_of(x, min), v)) {
                    val_out[i] = v;
                    r = true;
                }
            }
            out[i] = r;
        }
        return;
    }
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK) {
        bool r = false;
        if (in[i]) {
            const int32_t x = probe[i];
            int32_t v;
            if (x >= min && x <= max && probe_value(t, use16, vmin, slot_of(x, min), v)) {
                val_out[i] = v;
                r = true;
            }
        }
        out[i] = r;
    }
}

// Each block's min and max of the values of the slots whose flag is 1, to
// partials[2 b], [2 b + 1] (no slot set: INT32_MAX, INT32_MIN)
constexpr unsigned PAIRS_RANGE_BLOCKS = BLOCK; // one partial per thread of the reader

__global__ void __launch_bounds__(BLOCK) k_pairs_range(const int2 *__restrict__ pairs, int64_t len, int32_t *partials)
{
    int32_t lo = INT32_MAX, hi = INT32_MIN;
    for (int64_t base = (int64_t)blockIdx.x * BLOCK * UNROLL; base < len;
         base += (int64_t)gridDim.x * BLOCK * UNROLL) {
        int2 e[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            const int64_t h = base + u * BLOCK + threadIdx.x;
            e[u] = h < len ? pairs[h] : make_int2(0, 0);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; u++)
            if (e[u].x == 1) {
                lo = min(lo, e[u].y);
                hi = max(hi, e[u].y);
            }
    }
    block_minmax(lo, hi);
    if (threadIdx.x == 0) {
        partials[2 * blockIdx.x] = lo;
        partials[2 * blockIdx.x + 1] = hi;
    }
}

// The 16-bit copy and the presence bitmap of the pairs, 64 slots per wave and
// step (a wave's ballot gives two bitmap words).  Every block first reduces
// the partial ranges; block 0 leaves the result in info for the probe.
__global__ void __launch_bounds__(BLOCK) k_pairs_to_u16(const int2 *__restrict__ pairs, int64_t len,
                                                        const int32_t *__restrict__ partials, int nparts,
                                                        int32_t *info, uint16_t *u16, uint32_t *bits)
{
    __shared__ int32_t range[2];
    int32_t lo = INT32_MAX, hi = INT32_MIN;
    if ((int)threadIdx.x < nparts) {
        lo = partials[2 * threadIdx.x];
        hi = partials[2 * threadIdx.x + 1];
    }
    block_minmax(lo, hi);
    if (threadIdx.x == 0) {
        range[0] = lo;
        range[1] = hi;
    }
    __syncthreads();
    const int32_t vmin = range[0];
    // every value offset must stay below VALS_UNSET
    const bool fits = range[1] < vmin || (int64_t)range[1] - (int64_t)vmin < (int64_t)VALS_UNSET;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        info[0] = vmin;
        info[1] = range[1];
        info[2] = fits ? 0 : 1;
    }
    const int lane = threadIdx.x & 63;
    const int64_t words = (len + 31) / 32, nwaves = (int64_t)gridDim.x * (BLOCK / 64);
    for (int64_t g = (int64_t)blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6); g * 64 < len; g += nwaves) {
        const int64_t h = g * 64 + lane;
        const int2 e = h < len ? pairs[h] : make_int2(0, 0);
        if (fits && h < len) u16[h] = e.x == 1 ? (uint16_t)(e.y - vmin) : (uint16_t)VALS_UNSET;
        const uint64_t m = __ballot(e.x == 1);
        if (lane < 2 && 2 * g + lane < words) bits[2 * g + lane] = (uint32_t)(m >> (32 * lane));
    }
}

// The full probe of a long column against a table much smaller than it.  The
// table's gathers are the bound: 268M of them into a 2.8 MB 16-bit table cost
// 1.4 ms of 1.7 (each brings an L2 line for two bytes), against 0.35 ms for
// the column and the flags.  So the block keeps in LDS (one 1024-thread block
// per CU, 16 waves)
//   VALS  the whole 16-bit table, up to PROBE_LDS_SLOTS slots;
//   else  the presence bitmap, folded modulo the power of two that fits 128
//         KB: a clear bit settles the row, and only the rows that pass (the
//         matches and, folded, a few more) are listed and gather from the
//         table, up to 256 of them in flight per wave.
// 268M rows, 1.4M slots of which 4 % match, every row flagged: 1712 -> 712 us
// (the scattered value stores are most of the rest); 60M rows, 300,000 slots,
// 20 %: 374 -> 197 us; 61,130 slots in LDS, 0.8 % of 268M rows flagged: 340 ->
// 237 us.  The column, flags and touched value lines alone take 600 / 180 /
// 210 us at the rate of a copy.  Tiles go round the blocks wave by wave: with a
// block's waves on neighbouring tiles the last round kept some CUs busy and left
// the others idle (60M rows, 0.5 % flagged, 65,537 slots: 60 us so, 56 now; 20 %
// flagged, 300,000 slots: 194 and 181).  A table whose values need 32 bits is
// read in memory by half the waves of k_probe_full: 4M rows, 2,556 slots 33 us
// against 26, 60M rows 266 against 290.
constexpr int PROBE_BLOCK = 1024;
constexpr int64_t PROBE_LDS_SLOTS = 65536;        // 128 KB of 16-bit values
constexpr uint32_t PROBE_FILTER_WORDS = 1u << 15; // 128 KB of presence bits
constexpr int64_t PROBE_FILTER_SLOTS = 1 << 21;   // a listed row: slot and offset in its tile in 32 bits
constexpr uint32_t PROBE_OFF_BITS = 11;
static_assert(WT_ROWS == 1 << PROBE_OFF_BITS, "offset of a listed row");
constexpr uint32_t PROBE_LIST_MIN = 256;          // listed rows per wave: a chunk of the tile at least
constexpr uint32_t PROBE_LIST_MAX = 1024;
constexpr int PROBE_DRAIN = 4;

// Listed rows per wave beside a filter of `fwords` words (and a row mask per lane)
constexpr uint32_t probe_list_cap(uint32_t fwords)
{
    const uint32_t per_wave = (LDS_PER_CU - 4 * fwords) / 4 / (PROBE_BLOCK / 64) - 64;
    return per_wave < PROBE_LIST_MAX ? per_wave : PROBE_LIST_MAX;
}
static_assert(probe_list_cap(PROBE_FILTER_WORDS) >= PROBE_LIST_MIN, "LDS of the largest filter and the lists");

template <bool VALS>
__global__ void __launch_bounds__(PROBE_BLOCK) k_probe_full_lds(const int32_t *__restrict__ probe, int32_t *val_out,
                                                                const uint8_t *in, uint8_t *out, int64_t n,
                                                                PairsOrU16 t, const uint32_t *__restrict__ bits,
                                                                uint32_t words, uint32_t fwords, uint32_t cap,
                                                                int32_t min, int32_t max)
{
    extern __shared__ uint4 probe_lds[];
    const bool use16 = t.info[2] == 0;
    const int32_t vmin = t.info[0];
    const uint32_t span = (uint32_t)max - (uint32_t)min;
    if constexpr (VALS) {
        if (use16) // the 16-bit table (16-byte aligned and padded)
            for (uint32_t i = threadIdx.x; i < (span + 8u) / 8u; i += PROBE_BLOCK)
                probe_lds[i] = reinterpret_cast<const uint4 *>(t.u16)[i];
    } else {
        uint32_t *filter = reinterpret_cast<uint32_t *>(probe_lds);
        for (uint32_t d = threadIdx.x; d < fwords; d += PROBE_BLOCK) {
            uint32_t w = 0;
            for (uint32_t k = d; k < words; k += fwords) w |= bits[k];
            filter[d] = w;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    // scalar addresses save the filter's form 11 spilled registers (719 -> 705
    // us); the value table's form spills none and ran slower with them (233 -> 250)
    const int wave = VALS ? (int)(threadIdx.x >> 6) : wave_index();
    // the wave's row masks and list, behind the filter
    uint32_t *const hit_of = reinterpret_cast<uint32_t *>(probe_lds) + fwords + wave * (64 + cap);
    uint32_t *const list = hit_of + 64;
    const int64_t ntiles = n / WT_ROWS, stride = (int64_t)gridDim.x * (PROBE_BLOCK / 64);
    // (a last round is shared by all blocks)
    int64_t tile = blockIdx.x + (int64_t)gridDim.x * wave;
    uint32_t next[WT_CHUNKS];
    if (tile < ntiles) wt_flags(in, tile * WT_ROWS, lane, next);
    for (; tile < ntiles; tile += stride) {
        const int64_t t0 = tile * WT_ROWS;
        const uint32_t flagged = wt_mask(next);
        uint32_t other = 0; // flags other than 0 and 1 become 1
#pragma unroll
        for (int j = 0; j < WT_CHUNKS; j++) other |= next[j] & 0xfefefefeu;
        const bool odd = other != 0;
        uint32_t slot[WT_CHUNKS][4];
#pragma unroll
        for (int j = 0; j < WT_CHUNKS; j++) {
            int4 x = make_int4(0, 0, 0, 0);
            if ((flagged >> (4 * j)) & 15u) x = *reinterpret_cast<const int4 *>(probe + wt_row(t0, lane, j));
            slot[j][0] = (uint32_t)x.x - (uint32_t)min;
            slot[j][1] = (uint32_t)x.y - (uint32_t)min;
            slot[j][2] = (uint32_t)x.z - (uint32_t)min;
            slot[j][3] = (uint32_t)x.w - (uint32_t)min;
        }
        // the next tile's flags load while this one is probed
        if (tile + stride < ntiles) wt_flags(in, t0 + stride * WT_ROWS, lane, next);
        uint32_t cand = 0;
#pragma unroll
        for (int b = 0; b < 4 * WT_CHUNKS; b++) {
            const uint32_t s = slot[b >> 2][b & 3];
            bool go = s <= span;
            if constexpr (!VALS) {
                const uint32_t *filter = reinterpret_cast<const uint32_t *>(probe_lds);
                go &= ((filter[(s >> 5) & (fwords - 1)] >> (s & 31)) & 1u) != 0;
            }
            cand |= (uint32_t)go << b;
        }
        cand &= flagged;
        uint32_t hits = 0;
        if (!VALS && use16) {
            if constexpr (!VALS) {
                uint32_t total;
                uint32_t at = wave_prefix((uint32_t)__popc(cand), lane, total);
                hit_of[lane] = 0;
                // a list too short for the tile takes a chunk (256 rows) at a time
                const bool one = total <= cap;
                uint32_t count = total;
#pragma unroll
                for (int j = 0; j < WT_CHUNKS; j++) {
                    if (!one) at = wave_prefix((uint32_t)__popc((cand >> (4 * j)) & 15u), lane, count);
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        if ((cand >> (4 * j + k)) & 1u)
                            list[at++] = slot[j][k] << PROBE_OFF_BITS | wt_offset(lane, 4 * j + k);
                    if (one && j + 1 < WT_CHUNKS) continue;
                    wave_sync();
                    for (uint32_t e = 0; e < count; e += 64 * PROBE_DRAIN) {
                        uint32_t v[PROBE_DRAIN], o[PROBE_DRAIN];
#pragma unroll
                        for (int d = 0; d < PROBE_DRAIN; d++) {
                            const uint32_t i = e + 64 * d + lane;
                            v[d] = VALS_UNSET;
                            if (i < count) {
                                o[d] = list[i];
                                v[d] = t.u16[o[d] >> PROBE_OFF_BITS];
                            }
                        }
#pragma unroll
                        for (int d = 0; d < PROBE_DRAIN; d++) {
                            if (v[d] == VALS_UNSET) continue;
                            o[d] &= (1u << PROBE_OFF_BITS) - 1;
                            val_out[t0 + o[d]] = vmin + (int32_t)v[d];
                            atomicOr(&hit_of[(o[d] >> 2) & 63u], 1u << ((o[d] >> 8) * 4 + (o[d] & 3u)));
                        }
                    }
                    wave_sync();
                }
                hits = hit_of[lane];
                wave_sync();
            }
        } else {
#pragma unroll
            for (int j = 0; j < WT_CHUNKS; j++) {
                if (!((cand >> (4 * j)) & 15u)) continue;
                const int64_t r = wt_row(t0, lane, j);
                int32_t v[4];
                uint32_t hit = 0;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    if (!((cand >> (4 * j + k)) & 1u)) continue;
                    if (VALS && use16) {
                        const uint32_t raw = reinterpret_cast<const uint16_t *>(probe_lds)[slot[j][k]];
                        v[k] = vmin + (int32_t)raw;
                        hit |= (uint32_t)(raw != VALS_UNSET) << k;
                    } else {
                        const int2 e = t.pairs[slot[j][k]];
                        v[k] = e.y;
                        hit |= (uint32_t)(e.x == 1) << k;
                    }
                }
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if ((hit >> k) & 1u) val_out[r + k] = v[k];
                hits |= hit << (4 * j);
            }
        }
#pragma unroll
        for (int j = 0; j < WT_CHUNKS; j++) {
            const int64_t r = wt_row(t0, lane, j);
            const uint32_t f = flag_bytes(hits >> (4 * j));
            // in place, flags that stay as they are need no write
            if (in == out && !__any(odd || (((hits ^ flagged) >> (4 * j)) & 15u))) continue;
            *reinterpret_cast<uint32_t *>(out + r) = f;
        }
    }
    if (blockIdx.x + 1 == gridDim.x)
        for (int64_t i = ntiles * WT_ROWS + threadIdx.x; i < n; i += PROBE_BLOCK) {
            const uint32_t s = (uint32_t)probe[i] - (uint32_t)min;
            bool hit = false;
            if (in[i] && s <= span) {
                int32_t v;
                if (use16) {
                    const uint32_t raw = VALS ? reinterpret_cast<const uint16_t *>(probe_lds)[s] : t.u16[s];
                    v = vmin + (int32_t)raw;
                    hit = raw != VALS_UNSET;
                } else {
                    const int2 e = t.pairs[s];
                    v = e.y;
                    hit = e.x == 1;
                }
                if (hit) val_out[i] = v;
            }
            out[i] = hit;
        }
}

// ----------------------------------------------------------- aggregation

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        v += __shfl_xor(v, off, 64);
    return v;
}

// The scalar reductions run 1024-thread blocks, at most two per CU: each block
// ends in one atomic on the same word, and those serialise at about 10 ns
// each.  With 2,048 blocks of 256 threads they took a third of a 60M-row sum
// and half of a 100M-row count (sum with 2 % of
// the rows flagged 54 -> 36 us, count 51 -> 22 us).
constexpr int RED_BLOCK = 1024;
constexpr int RED_PER_CU = 2;

// Block-wide sum; one atomic per block into *acc.
__device__ __forceinline__ void block_add_u64(uint64_t v, uint64_t *acc)
{
    __shared__ uint64_t part[RED_BLOCK / 64];
    v = wave_sum_u64(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) part[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t s = 0;
#pragma unroll
        for (int w = 0; w < RED_BLOCK / 64; w++) s += part[w];
        if (s) atomicAdd(reinterpret_cast<unsigned long long *>(acc), (unsigned long long)s);
    }
}

__global__ void __launch_bounds__(RED_BLOCK) k_sum_flagged(const int32_t *__restrict__ col,
                                                       const uint8_t *__restrict__ flags, int64_t n,
                                                       uint64_t *acc, int vec)
{
    int64_t s = 0; // int64 partial; the uint64 total is its two's-complement image
    if (vec) {
        const int64_t nchunks = n >> 2;
        const int4 *c4 = reinterpret_cast<const int4 *>(col);
        const uint32_t *f32 = reinterpret_cast<const uint32_t *>(flags);
        for (int64_t base = (int64_t)blockIdx.x * RED_BLOCK * UNROLL; base < nchunks;
             base += (int64_t)gridDim.x * RED_BLOCK * UNROLL) {
            uint32_t f[UNROLL];
            int4 x[UNROLL];
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                const int64_t c = base + u * RED_BLOCK + threadIdx.x;
                f[u] = c < nchunks ? f32[c] : 0u;
                if (f[u]) x[u] = c4[c];
            }
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                if (!f[u]) continue;
                s += byte_of(f[u], 0) ? (int64_t)x[u].x : 0;
                s += byte_of(f[u], 1) ? (int64_t)x[u].y : 0;
                s += byte_of(f[u], 2) ? (int64_t)x[u].z : 0;
                s += byte_of(f[u], 3) ? (int64_t)x[u].w : 0;
            }
        }
        if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {
            const int64_t i = (nchunks << 2) + threadIdx.x;
            if (flags[i]) s += col[i];
        }
    } else {
        for (int64_t i = (int64_t)blockIdx.x * RED_BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * RED_BLOCK)
            if (flags[i]) s += col[i];
    }
    block_add_u64((uint64_t)s, acc);
}

// 16 flags per load, at any alignment (200M flags 4 bytes past an aligned start:
// 130 us one by one, 63 four at a time where aligned to 4, 35 so).
__global__ void __launch_bounds__(RED_BLOCK) k_count_flags(const uint8_t *flags, int64_t n, uint64_t *acc)
{
    uint64_t s = 0;
    const int64_t nq = n >> 4;
    for (int64_t base = (int64_t)blockIdx.x * RED_BLOCK * UNROLL; base < nq;
         base += (int64_t)gridDim.x * RED_BLOCK * UNROLL) {
        uint4 q[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; u++) {
            const int64_t c = base + u * RED_BLOCK + threadIdx.x;
            q[u] = make_uint4(0, 0, 0, 0);
            if (c < nq) __builtin_memcpy(&q[u], flags + 16 * c, 16);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; u++)
            s += __popc(nz_bytes(q[u].x)) + __popc(nz_bytes(q[u].y)) + __popc(nz_bytes(q[u].z)) + __popc(nz_bytes(q[u].w));
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 15)) s += flags[(nq << 4) + threadIdx.x] != 0;
    block_add_u64(s, acc);
}

constexpr int GB_MAX_KEYS = 8;
struct GroupArgs {
    const int32_t *keys[GB_MAX_KEYS];
    int32_t *out_keys[GB_MAX_KEYS];
    int32_t mins[GB_MAX_KEYS];
    int32_t maxs[GB_MAX_KEYS];
    uint32_t range[GB_MAX_KEYS]; // max - min + 1 (uint32 image of the int)
    int k;
};

// Dense slot of row i exactly as GroupByAggregateKernel computes it
// (int32 wrapping accumulation, then % prod on the uint64 image).
__device__ __forceinline__ uint32_t group_slot(const GroupArgs &g, const int32_t *kv, uint64_t prod)
{
    uint32_t hash = 0, mult = 1;
    for (int j = 0; j < g.k; j++) {
        hash += ((uint32_t)kv[j] - (uint32_t)g.mins[j]) * mult;
        mult *= g.range[j];
    }
    const uint64_t h64 = (uint64_t)(int64_t)(int32_t)hash;
    return (uint32_t)(h64 % prod);
}

// Global path: one exchange + one atomic add per flagged row.
__device__ __forceinline__ void group_row_global(const GroupArgs &g, const int32_t *kv, int32_t agg,
                                                 uint64_t *sums, uint32_t *seen, uint64_t prod)
{
    const uint32_t s = group_slot(g, kv, prod);
    if (atomicExch(&seen[s], 1u) == 0u)
        for (int j = 0; j < g.k; j++) g.out_keys[j][s] = kv[j];
    atomicAdd(reinterpret_cast<unsigned long long *>(&sums[s]), (unsigned long long)(int64_t)agg);
}

__global__ void __launch_bounds__(BLOCK) k_groupby_global(GroupArgs g, const int32_t *agg,
                                                          const uint8_t *flags, int64_t n,
                                                          uint64_t *sums, uint32_t *seen, uint64_t prod)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK) {
        if (!flags[i]) continue;
        int32_t kv[GB_MAX_KEYS];
        for (int j = 0; j < g.k; j++) kv[j] = g.keys[j][i];
        group_row_global(g, kv, agg[i], sums, seen, prod);
    }
}

// LDS-privatised dense group-by: each block accumulates its rows into an LDS
// copy of the dense sum array (ds_add_u64) plus an occupancy bitmap, then
// flushes the occupied slots with one global atomic each.  Rows whose keys
// all lie in [min, max] map to a unique slot whose key values are recovered
// from the slot index at flush; any other row takes the global path so the
// key it stores is its own.
//
// A wave lists the flagged rows of its tile in LDS and takes them from there
// 64 x GB_DRAIN at a time, one row per lane and step: the keys and values of
// up to 256 rows are then in flight together.  Taking them where they lie
// instead (each lane its own rows) costs a round trip to memory per row slot
// that any lane of the wave has flagged, nearly all of them already at 1 % of
// the rows (2^28 rows, 0.8 % flagged, 7,000 slots: 736 -> 189 us;
// 60M rows, 1.6 %, 175 slots: 274 -> 70 us; every row flagged, three keys of
// 4,375 slots: 514 -> 200 us).
constexpr int GB_BLOCK = 1024; // threads per block of the LDS group-by
constexpr int GB_DRAIN = 4;
constexpr uint32_t GB_LIST = 512; // listed rows per wave: two of a dense tile's chunks

// K: number of keys (0: g.k, up to GB_MAX_KEYS)
template <int K>
__global__ void __launch_bounds__(GB_BLOCK) k_groupby_lds(GroupArgs g, const int32_t *agg, const uint8_t *flags,
                                                          int64_t n, uint64_t *sums, uint32_t *seen, uint32_t prod)
{
    extern __shared__ unsigned long long lds[];
    __shared__ uint16_t lists[GB_BLOCK / 64][GB_LIST];
    constexpr int KMAX = K ? K : GB_MAX_KEYS;
    const int nk = K ? K : g.k;
    unsigned long long *lsum = lds;
    uint32_t *lbits = reinterpret_cast<uint32_t *>(lds + prod);
    const uint32_t nwords = (prod + 31) / 32;
    for (uint32_t s = threadIdx.x; s < prod; s += GB_BLOCK) lsum[s] = 0;
    for (uint32_t w = threadIdx.x; w < nwords; w += GB_BLOCK) lbits[w] = 0;
    __syncthreads();
    auto take = [&](const int32_t (&kv)[KMAX], int32_t v) {
        bool in_range = true;
        uint32_t s = 0, mult = 1;
#pragma unroll
        for (int j = 0; j < KMAX; j++)
            if (j < nk) {
                in_range &= kv[j] >= g.mins[j] && kv[j] <= g.maxs[j];
                s += ((uint32_t)kv[j] - (uint32_t)g.mins[j]) * mult;
                mult *= g.range[j];
            }
        if (!in_range) {
            group_row_global(g, kv, v, sums, seen, prod);
            return;
        }
        // in range, s is below prod (the ranges multiply to it)
        atomicAdd(&lsum[s], (unsigned long long)(int64_t)v);
        if (!((lbits[s >> 5] >> (s & 31)) & 1u)) atomicOr(&lbits[s >> 5], 1u << (s & 31));
    };
    const int lane = threadIdx.x & 63;
    uint16_t *list = lists[threadIdx.x >> 6];
    const int64_t ntiles = n / WT_ROWS, stride = (int64_t)gridDim.x * (GB_BLOCK / 64);
    int64_t t = (int64_t)blockIdx.x * (GB_BLOCK / 64) + (threadIdx.x >> 6);
    uint32_t next[WT_CHUNKS];
    if (t < ntiles) wt_flags(flags, t * WT_ROWS, lane, next);
    for (; t < ntiles; t += stride) {
        const int64_t t0 = t * WT_ROWS;
        const uint32_t tile = wt_mask(next);
        // the next tile's flags load while this one's rows are taken
        if (t + stride < ntiles) wt_flags(flags, t0 + stride * WT_ROWS, lane, next);
        uint32_t total;
        uint32_t at = wave_prefix((uint32_t)__popc(tile), lane, total);
        const int parts = total <= GB_LIST ? 1 : 4;
        for (int part = 0; part < parts; part++) {
            uint32_t m = tile, count = total;
            if (parts > 1) {
                m = (tile >> (8 * part)) & 0xffu;
                at = wave_prefix((uint32_t)__popc(m), lane, count);
            }
            for (; m; m &= m - 1) list[at++] = (uint16_t)wt_offset(lane, (uint32_t)__builtin_ctz(m) + 8u * part);
            wave_sync();
            for (uint32_t e = 0; e < count; e += 64 * GB_DRAIN) {
                // (lanes past the list read its last row again: loads under
                // a condition of their own waited for each other)
                int32_t kv[GB_DRAIN][KMAX], v[GB_DRAIN];
                uint32_t o[GB_DRAIN];
#pragma unroll
                for (int d = 0; d < GB_DRAIN; d++) o[d] = list[min(e + 64 * d + lane, count - 1)];
#pragma unroll
                for (int d = 0; d < GB_DRAIN; d++) {
                    const int64_t row = t0 + o[d];
#pragma unroll
                    for (int j = 0; j < KMAX; j++)
                        if (j < nk) kv[d][j] = g.keys[j][row];
                    v[d] = agg[row];
                }
#pragma unroll
                for (int d = 0; d < GB_DRAIN; d++)
                    if (e + 64 * d + lane < count) take(kv[d], v[d]);
            }
            wave_sync();
        }
    }
    if (blockIdx.x + 1 == gridDim.x)
        for (int64_t i = ntiles * WT_ROWS + threadIdx.x; i < n; i += GB_BLOCK) {
            if (!flags[i]) continue;
            int32_t kv[KMAX];
#pragma unroll
            for (int j = 0; j < KMAX; j++)
                if (j < nk) kv[j] = g.keys[j][i];
            take(kv, agg[i]);
        }
    __syncthreads();
    for (uint32_t s = threadIdx.x; s < prod; s += GB_BLOCK) {
        if (!((lbits[s >> 5] >> (s & 31)) & 1u)) continue;
        atomicAdd(reinterpret_cast<unsigned long long *>(&sums[s]), lsum[s]);
        if (atomicExch(&seen[s], 1u) == 0u) {
            uint32_t rest = s;
            for (int j = 0; j < nk; j++) {
                g.out_keys[j][s] = (int32_t)((uint32_t)g.mins[j] + rest % g.range[j]);
                rest /= g.range[j];
            }
        }
    }
}

__global__ void __launch_bounds__(BLOCK) k_seen_to_flags(const uint32_t *seen, uint8_t *flags, uint64_t prod)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < (int64_t)prod; i += (int64_t)gridDim.x * BLOCK)
        flags[i] = seen[i] != 0;
}

// ------------------------------------------------------ compact probe tables
// Deterministic (no atomics on the tables).  The population count is left
// per block and summed when the statistics are read (k_stats_reduce).

// Stores the block's count (the sum of every wave's, held by its lane 0) in
// *count.  One same-address atomic per block instead
// serialises: 1,368 blocks over the 1.4M-slot part table took 21 us, 7 us
// with the partial counts.
__device__ __forceinline__ void block_count_store(uint32_t local, uint32_t *count)
{
    __shared__ uint32_t wave_sum[BLOCK / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) wave_sum[wave] = local;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
#pragma unroll
        for (int w = 0; w < BLOCK / 64; w++) t += wave_sum[w];
        *count = t;
    }
}

// Presence bitmaps of the reference tables: one thread per slot, each wave
// covering 64 consecutive slots (coalesced reads), its ballot giving two
// bitmap words; the set slots are counted per wave, then per block (one
// partial count per block, bits_partials(len) of them).
// Each wave takes BITS_GROUPS consecutive 64-slot groups per step, their
// loads issued together, on a grid of at most BITS_MAX_BLOCKS blocks.  From
// the pairs, the 16-bit value table is written too: value - vmin in the set
// slots, VALS_UNSET in the others (`bad` is raised when a set slot's offset
// does not fit below VALS_UNSET, and the table is then not used).
constexpr int BITS_GROUPS = 4;
constexpr unsigned BITS_MAX_BLOCKS = 2048;

// tables per launch (their descriptions are kernel arguments: the small form
// for one plan's joins, the large one for a batch's)
constexpr int COMPACT_JOBS_SMALL = 4, COMPACT_JOBS = 32;
struct BitsJob {
    const void *ht;
    uint32_t *bits;
    uint16_t *vals;
    uint32_t *partials, *bad;
    int32_t len, vmin;
    uint32_t nblocks, pairs;
};
template <int N> struct BitsJobs {
    uint32_t first[N];
    BitsJob job[N];
};
struct RankJob {
    const uint32_t *bits, *partials;
    const uint16_t *vals;
    uint8_t *dict;
    int32_t len, words;
    uint32_t cap_vals;
};
template <int N> struct RankJobs {
    uint32_t first[N];
    RankJob job[N];
};
static_assert(sizeof(BitsJobs<COMPACT_JOBS>) <= 4096 && sizeof(RankJobs<COMPACT_JOBS>) <= 4096, "kernel argument segment");

__device__ __forceinline__ void bits_from_keys(const BitsJob &J, uint32_t block, uint32_t nblocks)
{
    const uint8_t *ht = static_cast<const uint8_t *>(J.ht);
    const int64_t len = J.len, words = (len + 31) / 32;
    const int lane = threadIdx.x & 63;
    const int64_t nwaves = ((int64_t)nblocks * BLOCK) >> 6;
    uint32_t local = 0;
    for (int64_t g0 = (((int64_t)block * BLOCK + threadIdx.x) >> 6) * BITS_GROUPS; g0 * 64 < len;
         g0 += nwaves * BITS_GROUPS) {
        bool set[BITS_GROUPS];
#pragma unroll
        for (int k = 0; k < BITS_GROUPS; k++) {
            const int64_t s = (g0 + k) * 64 + lane;
            set[k] = s < len && ht[s] != 0;
        }
#pragma unroll
        for (int k = 0; k < BITS_GROUPS; k++) {
            const int64_t g = g0 + k;
            const uint64_t m = __ballot(set[k]);
            if (lane == 0 && 2 * g < words) {
                J.bits[2 * g] = (uint32_t)m;
                if (2 * g + 1 < words) J.bits[2 * g + 1] = (uint32_t)(m >> 32);
                local += (uint32_t)__popcll(m);
            }
        }
    }
    block_count_store(local, J.partials + block);
}

__device__ __forceinline__ void bits_from_pairs(const BitsJob &J, uint32_t block, uint32_t nblocks)
{
    const int2 *ht = static_cast<const int2 *>(J.ht);
    uint16_t *vals = J.vals;
    const int64_t len = J.len, words = (len + 31) / 32;
    const int lane = threadIdx.x & 63;
    const int64_t nwaves = ((int64_t)nblocks * BLOCK) >> 6;
    uint32_t local = 0;
    bool ok = true;
    for (int64_t g0 = (((int64_t)block * BLOCK + threadIdx.x) >> 6) * BITS_GROUPS; g0 * 64 < len;
         g0 += nwaves * BITS_GROUPS) {
        int2 e[BITS_GROUPS];
#pragma unroll
        for (int k = 0; k < BITS_GROUPS; k++) {
            const int64_t s = (g0 + k) * 64 + lane;
            e[k] = s < len ? ht[s] : make_int2(0, 0);
        }
#pragma unroll
        for (int k = 0; k < BITS_GROUPS; k++) {
            const int64_t g = g0 + k, s = g * 64 + lane;
            const bool set = e[k].x == 1;
            // unset slots hold VALS_UNSET; a set slot's offset must stay below it
            const uint32_t d = set ? (uint32_t)e[k].y - (uint32_t)J.vmin : VALS_UNSET;
            ok &= !set || d < VALS_UNSET;
            if (vals && s < len) vals[s] = (uint16_t)d;
            const uint64_t m = __ballot(set);
            if (lane == 0 && 2 * g < words) {
                J.bits[2 * g] = (uint32_t)m;
                if (2 * g + 1 < words) J.bits[2 * g + 1] = (uint32_t)(m >> 32);
                local += (uint32_t)__popcll(m);
            }
        }
    }
    block_count_store(local, J.partials + block);
    if (!ok) atomicOr(J.bad, 1u);
}

// Several tables in one launch: block b works on the job whose blocks
// [first[j], first[j + 1]) hold it (unused entries of first: UINT32_MAX).
// A launch of 3 to 5 us per table, one after another, made up most of a small
// query's device time.
template <int N> __device__ __forceinline__ int job_of(const uint32_t (&first)[N], uint32_t block)
{
    int j = 0;
#pragma unroll
    for (int k = 1; k < N; k++) j += block >= first[k];
    return j;
}

template <int N> __global__ void __launch_bounds__(BLOCK) k_compact_bits(BitsJobs<N> jobs)
{
    const int j = job_of(jobs.first, blockIdx.x);
    const BitsJob &J = jobs.job[j];
    const uint32_t block = blockIdx.x - jobs.first[j];
    if (J.pairs) bits_from_pairs(J, block, J.nblocks);
    else bits_from_keys(J, block, J.nblocks);
}

// The windows of 32 consecutive keys (one bitmap word) of a table of WB-byte
// windows (1, 2 or 4 bytes), 16-byte aligned and padded to 16 bytes, in
// 2 * WB vector loads issued together.
template <uint32_t WB> struct DictWord {
    static constexpr uint32_t NQ = 2 * WB; // 16-byte chunks per 32 windows
    static constexpr uint32_t FIELD = WB >= 4 ? ~0u : (1u << (8u * (WB % 4u))) - 1u;
    uint4 q[NQ];
    // the windows of keys [32 w, 32 w + 32) that are below len; a chunk that
    // starts past the table's last window is not read
    __device__ __forceinline__ void load(const uint8_t *tab, uint32_t len, uint32_t w)
    {
        const uint4 *p = reinterpret_cast<const uint4 *>(tab) + (size_t)w * NQ;
        const uint32_t nbytes = min(len - w * 32u, 32u) * WB;
#pragma unroll
        for (uint32_t k = 0; k < NQ; k++) q[k] = 16u * k < nbytes ? p[k] : make_uint4(0u, 0u, 0u, 0u);
    }
    __device__ __forceinline__ uint32_t window(uint32_t e) const // e: compile-time after unrolling
    {
        const uint32_t byte = e * WB, k = byte >> 4, j = (byte >> 2) & 3u;
        const uint32_t c = j == 0 ? q[k].x : j == 1 ? q[k].y : j == 2 ? q[k].z : q[k].w;
        return (c >> (8u * (byte & 3u))) & FIELD;
    }
    __device__ __forceinline__ uint32_t bits(uint32_t len, uint32_t w) const
    {
        uint32_t m = 0;
#pragma unroll
        for (uint32_t e = 0; e < 32u; e++) m |= (uint32_t)(window(e) != 0u) << e;
        const uint32_t n = min(len - w * 32u, 32u);
        return n == 32u ? m : m & ((1u << n) - 1u);
    }
    // the windows of the keys set in m, at ranks rank, rank + 1, ... (those
    // at or past cap are dropped)
    template <class T> __device__ __forceinline__ void write(uint32_t m, uint32_t rank, T *vals, uint32_t cap) const
    {
#pragma unroll
        for (uint32_t e = 0; e < 32u; e++)
            if ((m >> e) & 1u) {
                if (rank < cap) vals[rank] = (T)window(e);
                rank++;
            }
    }
};

// Rank dictionary of a presence bitmap with per-slot 16-bit values (the
// layout FV_RANK16 describes in fused_types.hpp), from the per-block counts
// of bits_from_pairs: its block b counted exactly the slots
// [1024 b, 1024 b + 1024), i.e. the bitmap words [32 b, 32 b + 32).  One wave
// per such range: its set slots before the range are the partial counts of
// the blocks before it; lane l < 32 takes word 32 b + l, the wave scans the
// words' counts, and each lane writes its word, its prefix and its set
// slots' values (four vector loads issued together).
constexpr uint32_t RANK_PART_WORDS = 32;

template <int N> __global__ void __launch_bounds__(64) k_rank_dicts(RankJobs<N> jobs)
{
    const int j = job_of(jobs.first, blockIdx.x);
    const RankJob &J = jobs.job[j];
    const uint32_t *bits = J.bits, *partials = J.partials;
    const int32_t words = J.words;
    uint8_t *dict = J.dict;
    const int lane = threadIdx.x;
    const uint32_t b = blockIdx.x - jobs.first[j];
    const int32_t w = (int32_t)(b * RANK_PART_WORDS) + (lane & 31);
    const uint32_t m = lane < 32 && w < words ? bits[w] : 0u;
    uint32_t before = 0;
    for (uint32_t i = lane; i < b; i += 64) before += partials[i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
    const uint32_t c = __popc(m);
    uint32_t incl = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(incl, off, 64);
        if (lane >= off) incl += y;
    }
    if (lane >= 32 || w >= words) return;
    const uint32_t base = before + incl - c;
    reinterpret_cast<uint32_t *>(dict)[w] = m;
    reinterpret_cast<uint16_t *>(dict + rank_prefix_off((uint32_t)words))[w] = (uint16_t)base;
    if (m) {
        DictWord<2> x;
        x.load(reinterpret_cast<const uint8_t *>(J.vals), (uint32_t)J.len, (uint32_t)w);
        x.write(m, base, reinterpret_cast<uint16_t *>(dict + rank_values_off((uint32_t)words)), J.cap_vals);
    }
}

// ------------------------------------------------------- batch probe masks
// Every key of a masked fact column: the key's word starts with every
// program's bit and loses the bit of each program one of whose probes on the
// column fails for the key -- the probe's own test (range check, then the
// table entry: FilterJoinKernel / FullJoinKernel, kernels/join.hpp:129-160,
// 256-300).
//
// Four consecutive keys per thread (their bits of a bitmap lie in one or two
// words, their windows in one store), 1,024 per block; the block's entries
// come through LDS, and the bitmap words of four entries load together.
constexpr uint32_t MASK_KEYS = 4 * BLOCK;
constexpr uint32_t MASK_ENTS = 64; // entries in LDS at a time
constexpr int MASK_GROUP = 4;
struct MaskGrid {
    uint32_t first[F_MASK_MAX_COLS]; // first block of each column (unused: UINT32_MAX)
};

// bit k: whether the probe passes for key + k
__device__ __forceinline__ uint32_t mask_probe(const FMaskEntry &E, int32_t key)
{
    uint32_t m = 0;
    for (int k = 0; k < 4; k++) {
        const int32_t x = (int32_t)((uint32_t)key + (uint32_t)k);
        if (x < E.ht_min || x > E.ht_max) continue;
        const uint32_t s = slot_of(x, E.ht_min);
        bool pass;
        if (E.kind == FM_BITS) pass = (reinterpret_cast<const uint32_t *>(E.ht)[s >> 5] >> (s & 31)) & 1u;
        else if (E.kind == FM_SEMI) pass = reinterpret_cast<const uint8_t *>(E.ht)[s] != 0;
        else pass = reinterpret_cast<const int2 *>(E.ht)[s].x == 1;
        m |= (uint32_t)pass << k;
    }
    return m;
}

__global__ void __launch_bounds__(BLOCK) k_batch_masks(const FMaskCol *__restrict__ cols,
                                                       const FMaskEntry *__restrict__ ents, MaskGrid grid)
{
    __shared__ FMaskEntry E[MASK_ENTS];
    int j = 0;
#pragma unroll
    for (int k = 1; k < F_MASK_MAX_COLS; k++) j += blockIdx.x >= grid.first[k];
    const FMaskCol c = cols[j];
    const uint32_t i = (blockIdx.x - grid.first[j]) * MASK_KEYS + 4u * threadIdx.x;
    const int32_t key = (int32_t)((uint32_t)c.lo + i);
    uint32_t w[4] = {c.full, c.full, c.full, c.full};
    for (uint32_t e0 = 0; e0 < c.count; e0 += MASK_ENTS) {
        const uint32_t n = min(c.count - e0, MASK_ENTS);
        __syncthreads();
        for (uint32_t e = threadIdx.x; e < n; e += BLOCK) E[e] = ents[c.first + e0 + e];
        __syncthreads();
        if (i >= c.len) continue;
        for (uint32_t e = 0; e < n; e += MASK_GROUP) {
            uint32_t lo[MASK_GROUP], hi[MASK_GROUP], slot[MASK_GROUP];
            bool whole[MASK_GROUP]; // a bitmap that holds all four keys
#pragma unroll
            for (int q = 0; q < MASK_GROUP; q++) {
                const uint32_t at = min(e + q, n - 1u);
                const uint32_t s = slot_of(key, E[at].ht_min), last = slot_of(E[at].ht_max, E[at].ht_min);
                whole[q] = E[at].kind == FM_BITS && E[at].ht_min <= E[at].ht_max && s <= last && last - s >= 3u;
                slot[q] = s;
                lo[q] = hi[q] = 0;
                if (whole[q]) {
                    const uint32_t *bits = reinterpret_cast<const uint32_t *>(E[at].ht);
                    lo[q] = bits[s >> 5];
                    hi[q] = bits[(s + 3u) >> 5];
                }
            }
#pragma unroll
            for (int q = 0; q < MASK_GROUP; q++) {
                if (e + q >= n) break;
                const uint32_t pass = whole[q] ? __builtin_amdgcn_alignbit(hi[q], lo[q], slot[q] & 31u)
                                               : mask_probe(E[e + q], key);
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (!((pass >> k) & 1u)) w[k] &= ~(1u << E[e + q].bit);
            }
        }
    }
    if (i >= c.len) return;
    // (the table is padded to 16 bytes: the last keys' windows store whole)
#pragma unroll
    for (int k = 0; k < 4; k++) w[k] >>= c.shift;
    if (c.wbytes == 1)
        *reinterpret_cast<uint32_t *>(c.tab + i) =
            (w[0] & 0xffu) | (w[1] & 0xffu) << 8 | (w[2] & 0xffu) << 16 | (w[3] & 0xffu) << 24;
    else if (c.wbytes == 2)
        *reinterpret_cast<uint2 *>(c.tab + 2 * i) = make_uint2((w[0] & 0xffffu) | w[1] << 16, (w[2] & 0xffffu) | w[3] << 16);
    else
        *reinterpret_cast<uint4 *>(c.tab + 4 * (size_t)i) = make_uint4(w[0], w[1], w[2], w[3]);
}

// Rank dictionaries of batched mask tables (FMaskDict), one block per table.
// Each thread takes whole bitmap words: the word's 32 windows (32 x 1, 2 or 4
// bytes, 16-byte aligned -- every table starts on 16 bytes and is padded to
// 16) come in with 2, 4 or 8 vector loads issued together, and the word's
// bit per key is whether the key's window is nonzero.  The exclusive counts
// before each word are scanned across the block; then each thread reloads its
// words' windows and writes every set key's window at its rank.
constexpr int DICT_BLOCK = 1024;
constexpr uint32_t DICT_MAX_WORDS = F_DICT_MAX_LEN / 32;

template <uint32_t WB> __device__ void dict_bits(const FMaskDict &d, uint32_t words, uint32_t *sbits)
{
    for (uint32_t w = threadIdx.x; w < words; w += DICT_BLOCK) {
        DictWord<WB> x;
        x.load(d.tab, d.len, w);
        sbits[w] = x.bits(d.len, w);
    }
}

template <uint32_t WB>
__device__ void dict_values(const FMaskDict &d, uint32_t words, const uint32_t *sbits, const uint32_t *spre,
                            uint32_t *vals)
{
    for (uint32_t w = threadIdx.x; w < words; w += DICT_BLOCK) {
        const uint32_t m = sbits[w];
        if (!m) continue;
        DictWord<WB> x;
        x.load(d.tab, d.len, w);
        x.write(m, spre[w], vals, ~0u);
    }
}

__global__ void __launch_bounds__(DICT_BLOCK) k_batch_dict(const FMaskDict *dicts)
{
    __shared__ uint32_t sbits[DICT_MAX_WORDS];
    __shared__ uint32_t spre[DICT_MAX_WORDS];
    __shared__ uint32_t wave_total[DICT_BLOCK / 64];
    const FMaskDict d = dicts[blockIdx.x];
    const uint32_t words = dict_words(d.len);
    if (d.wbytes == 1) dict_bits<1>(d, words, sbits);
    else if (d.wbytes == 2) dict_bits<2>(d, words, sbits);
    else dict_bits<4>(d, words, sbits);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t per = (words + DICT_BLOCK - 1) / DICT_BLOCK;
    const uint32_t a = min(words, threadIdx.x * per), b = min(words, a + per);
    uint32_t local = 0;
    for (uint32_t w = a; w < b; w++) local += __popc(sbits[w]);
    uint32_t incl = local;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(incl, off, 64);
        if (lane >= off) incl += y;
    }
    if (lane == 63) wave_total[wave] = incl;
    __syncthreads();
    uint32_t base = incl - local, total = 0;
    for (int v = 0; v < DICT_BLOCK / 64; v++) {
        if (v < wave) base += wave_total[v];
        total += wave_total[v];
    }
    for (uint32_t w = a; w < b; w++) {
        spre[w] = base;
        base += __popc(sbits[w]);
    }
    __syncthreads();
    uint32_t *hdr = reinterpret_cast<uint32_t *>(d.dict);
    uint32_t *obits = reinterpret_cast<uint32_t *>(d.dict + 16);
    uint16_t *opre = reinterpret_cast<uint16_t *>(d.dict + 16 + dict_prefix_off(d.len));
    uint32_t *ovals = reinterpret_cast<uint32_t *>(d.dict + 16 + dict_vals_off(d.len));
    for (uint32_t w = threadIdx.x; w < words; w += DICT_BLOCK) {
        obits[w] = sbits[w];
        opre[w] = (uint16_t)spre[w];
    }
    const bool ok = total <= F_DICT_CAP;
    if (ok) {
        if (d.wbytes == 1) dict_values<1>(d, words, sbits, spre, ovals);
        else if (d.wbytes == 2) dict_values<2>(d, words, sbits, spre, ovals);
        else dict_values<4>(d, words, sbits, spre, ovals);
    }
    if (threadIdx.x == 0) {
        hdr[0] = ok ? 1u : 0u;
        hdr[1] = total;
    }
}

// ------------------------------------------------------------ compaction
// Three passes over tiles of COMPACT_TILE rows, one wave per tile: count per
// tile, exclusive scan of the counts (one block), then write ids in row order.
// Flags come in 16 to a lane and load, at any alignment; a wave never waits for
// another one in the counting and writing passes (100M rows, one in twenty
// flagged: count 93 -> 18 us, scan 62 -> 6 us, write 181 -> 23 us; the count
// streams its flags at 5.7 TB/s).  A ragged end is read with the flags before
// it, in one load: byte by byte it cost a round trip each (200,001 rows 24 us,
// 17 so; 3M rows one byte past an aligned start 24.7 and 16).
constexpr int COMPACT_STEPS = 4; // steps of 64 lanes x 16 flags per tile
constexpr int64_t COMPACT_TILE = (int64_t)64 * 16 * COMPACT_STEPS;
constexpr int COMPACT_WAVES = BLOCK / 64; // tiles per block

// Bit k: whether byte k of q is nonzero.
__device__ __forceinline__ uint32_t nz_mask(const uint4 &q)
{
    return nz_mask(q.x) | nz_mask(q.y) << 4 | nz_mask(q.z) << 8 | nz_mask(q.w) << 12;
}

// Mask of the flags r .. r + 15 (at or past n: 0).
__device__ __forceinline__ uint32_t flags16(const uint8_t *flags, int64_t n, int64_t r)
{
    if (r >= n) return 0;
    const int64_t a = min(r, n - 16);
    if (a >= 0) {
        uint4 q;
        __builtin_memcpy(&q, flags + a, 16);
        return nz_mask(q) >> (int)(r - a);
    }
    uint32_t m = 0;
    for (int k = 0; r + k < n; k++) m |= (uint32_t)(flags[r + k] != 0) << k;
    return m;
}

// The flags of rows [t0 + 1024 u + 16 lane, ... + 16) as 16-bit masks; rows
// at or past n are 0.
__device__ __forceinline__ void tile_masks(const uint8_t *flags, int64_t n, int64_t t0, int lane,
                                           uint32_t (&m)[COMPACT_STEPS])
{
    if (t0 + COMPACT_TILE <= n) {
        uint4 q[COMPACT_STEPS];
#pragma unroll
        for (int u = 0; u < COMPACT_STEPS; u++) __builtin_memcpy(&q[u], flags + t0 + u * 1024 + lane * 16, 16);
#pragma unroll
        for (int u = 0; u < COMPACT_STEPS; u++) m[u] = nz_mask(q[u]);
        return;
    }
#pragma unroll
    for (int u = 0; u < COMPACT_STEPS; u++) {
        const int64_t r = t0 + u * 1024 + lane * 16;
        m[u] = flags16(flags, n, r);
    }
}

__global__ void __launch_bounds__(BLOCK) k_compact_count(const uint8_t *__restrict__ flags, int64_t n, int64_t ntiles,
                                                         uint32_t *__restrict__ counts)
{
    const int lane = threadIdx.x & 63;
    const int64_t t = (int64_t)blockIdx.x * COMPACT_WAVES + (threadIdx.x >> 6);
    if (t >= ntiles) return;
    uint32_t m[COMPACT_STEPS];
    tile_masks(flags, n, t * COMPACT_TILE, lane, m);
    uint32_t c = 0;
#pragma unroll
    for (int u = 0; u < COMPACT_STEPS; u++) c += __popc(m[u]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if (lane == 0) counts[t] = c;
}

// One block; a wave takes SCAN_VECS runs of 256 consecutive counts per step,
// four counts per lane and load.
constexpr int SCAN_BLOCK = 1024;
constexpr int SCAN_VECS = 4;

__global__ void __launch_bounds__(SCAN_BLOCK) k_compact_scan(uint32_t *counts, int64_t ntiles, uint32_t *count_out)
{
    __shared__ uint32_t wsum[2][SCAN_BLOCK / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool vec = ((uintptr_t)counts & 15) == 0;
    uint32_t carry = 0;
    int side = 0; // two copies of wsum: a step's writes never meet the last step's reads
    for (int64_t base = 0; base < ntiles; base += (int64_t)SCAN_BLOCK * SCAN_VECS * 4, side ^= 1) {
        const int64_t w0 = base + (int64_t)wave * 256 * SCAN_VECS;
        uint4 v[SCAN_VECS];
#pragma unroll
        for (int u = 0; u < SCAN_VECS; u++) {
            const int64_t t = w0 + u * 256 + lane * 4;
            if (vec && t + 3 < ntiles) v[u] = *reinterpret_cast<const uint4 *>(counts + t);
            else
                v[u] = make_uint4(t < ntiles ? counts[t] : 0u, t + 1 < ntiles ? counts[t + 1] : 0u,
                                  t + 2 < ntiles ? counts[t + 2] : 0u, t + 3 < ntiles ? counts[t + 3] : 0u);
        }
        uint32_t ex[SCAN_VECS], run = 0; // counts of the wave before the lane's vector u
#pragma unroll
        for (int u = 0; u < SCAN_VECS; u++) {
            uint32_t total;
            ex[u] = wave_prefix(v[u].x + v[u].y + v[u].z + v[u].w, lane, total) + run;
            run += total;
        }
        if (lane == 0) wsum[side][wave] = run;
        __syncthreads();
        uint32_t before = carry;
#pragma unroll
        for (int w = 0; w < SCAN_BLOCK / 64; w++) {
            if (w < wave) before += wsum[side][w];
            carry += wsum[side][w];
        }
#pragma unroll
        for (int u = 0; u < SCAN_VECS; u++) {
            const int64_t t = w0 + u * 256 + lane * 4;
            uint4 o;
            o.x = before + ex[u];
            o.y = o.x + v[u].x;
            o.z = o.y + v[u].y;
            o.w = o.z + v[u].z;
            if (vec && t + 3 < ntiles) *reinterpret_cast<uint4 *>(counts + t) = o;
            else {
                if (t < ntiles) counts[t] = o.x;
                if (t + 1 < ntiles) counts[t + 1] = o.y;
                if (t + 2 < ntiles) counts[t + 2] = o.z;
                if (t + 3 < ntiles) counts[t + 3] = o.w;
            }
        }
    }
    if (threadIdx.x == 0) *count_out = carry;
}

// A wave lists the selected rows of 1,024 flags in LDS and writes their ids from
// there 64 at a time; where all are selected it writes them at once.  (Taking
// the rows where they lie, 64 flags at a step, cost 900 instructions a tile
// whatever it held, and a store for every few rows: 100M rows, one in twenty
// flagged, 37 us against 25.)
__global__ void __launch_bounds__(BLOCK) k_compact_write(const uint8_t *__restrict__ flags, int64_t n, int64_t ntiles,
                                                         const uint32_t *__restrict__ offsets,
                                                         int32_t *__restrict__ row_ids)
{
    __shared__ uint16_t lists[COMPACT_WAVES][1024];
    const int lane = threadIdx.x & 63, wave = wave_index();
    const int64_t t = (int64_t)blockIdx.x * COMPACT_WAVES + wave;
    if (t >= ntiles) return;
    uint16_t *const list = lists[wave];
    const int64_t t0 = t * COMPACT_TILE;
    uint32_t m[COMPACT_STEPS];
    tile_masks(flags, n, t0, lane, m);
    int32_t *out = row_ids + offsets[t];
#pragma unroll
    for (int u = 0; u < COMPACT_STEPS; u++) {
        const int32_t r0 = (int32_t)(t0 + u * 1024);
        uint32_t total;
        uint32_t at = wave_prefix((uint32_t)__popc(m[u]), lane, total);
        if (total == 1024) {
#pragma unroll
            for (int i = 0; i < 1024; i += 64) out[i + lane] = r0 + i + lane;
        } else {
            for (uint32_t r = m[u]; r; r &= r - 1) list[at++] = (uint16_t)(16 * lane + __builtin_ctz(r));
            wave_sync();
            for (uint32_t i = lane; i < total; i += 64) out[i] = r0 + list[i];
            wave_sync();
        }
        out += total;
    }
}

__global__ void __launch_bounds__(BLOCK) k_gather_cols(GatherCols g, const int32_t *ids, int64_t count)
{
    for (int64_t j = (int64_t)blockIdx.x * BLOCK + threadIdx.x; j < count; j += (int64_t)gridDim.x * BLOCK) {
        const uint64_t r = (uint64_t)(uint32_t)ids[j];
        for (int c = 0; c < g.ncols; c++) {
            if ((g.is_u64 >> c) & 1u)
                static_cast<uint64_t *>(g.dst[c])[j] =
                    r < g.src_rows[c] ? static_cast<const uint64_t *>(g.src[c])[r] : 0ull;
            else
                static_cast<int32_t *>(g.dst[c])[j] = r < g.src_rows[c] ? static_cast<const int32_t *>(g.src[c])[r] : 0;
        }
    }
}

// blockIdx.y = part; the blocks of a part stride over its bytes (16 at a
// time where source and destination allow, the rest one by one).  One
// result's few parts come as a short argument list.
constexpr int PACK_FEW = 8;
template <int N> struct PackList {
    const uint8_t *src[N];
    uint64_t off[N];
    uint64_t bytes[N];
    uint8_t kind[N];
};

template <int N> __global__ void __launch_bounds__(BLOCK) k_pack_parts(PackList<N> p, uint8_t *dst)
{
    const int i = blockIdx.y;
    const uint8_t *src = p.src[i];
    const uint32_t *seen = reinterpret_cast<const uint32_t *>(src);
    uint8_t *out = dst + p.off[i];
    const uint64_t bytes = p.bytes[i];
    const uint32_t kind = p.kind[i];
    const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
    uint64_t head = 0;
    if ((((uintptr_t)src | (uintptr_t)out) & 15) == 0) {
        head = bytes & ~uint64_t(15);
        for (uint64_t j = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; j < head / 16; j += stride) {
            uint4 q = make_uint4(0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u);
            if (kind == PACK_COPY) q = reinterpret_cast<const uint4 *>(src)[j];
            else if (kind == PACK_SEEN) {
                uint32_t w[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint4 x = reinterpret_cast<const uint4 *>(seen)[4 * j + k];
                    w[k] = (uint32_t)(x.x != 0) | (uint32_t)(x.y != 0) << 8 | (uint32_t)(x.z != 0) << 16 |
                           (uint32_t)(x.w != 0) << 24;
                }
                q = make_uint4(w[0], w[1], w[2], w[3]);
            }
            reinterpret_cast<uint4 *>(out)[j] = q;
        }
    }
    for (uint64_t j = head + (uint64_t)blockIdx.x * BLOCK + threadIdx.x; j < bytes; j += stride)
        out[j] = kind == PACK_COPY ? src[j] : kind == PACK_SEEN ? (uint8_t)(seen[j] != 0) : (uint8_t)1;
}

// Selected rows of sparse result tables.  The rows cross PCIe where they are
// found: the host needs no count first, so it waits once and no gather,
// packing or transfer follows (the results of a 437,500-slot group-by took
// nine launches and two waits).  A tile is 2,048 rows, 8 per thread; the
// write pass adds up the tiles' counts before its own.
constexpr int SPARSE_TABLES = 8; // per launch
constexpr uint32_t SPARSE_TILE = 8 * BLOCK;
struct SparseJobs {
    uint32_t first[SPARSE_TABLES]; // first block of each table (unused: UINT32_MAX)
    SparseTable t[SPARSE_TABLES];
};
static_assert(sizeof(SparseJobs) <= 4096, "kernel argument segment");

__device__ __forceinline__ int sparse_job(const SparseJobs &jobs)
{
    int j = 0;
#pragma unroll
    for (int k = 1; k < SPARSE_TABLES; k++) j += blockIdx.x >= jobs.first[k];
    return j;
}

// bit k: row r + k is selected (r: a multiple of 8)
__device__ __forceinline__ uint32_t sparse_mask(const SparseTable &t, uint32_t r)
{
    uint32_t m = 0;
    if (r + 8u <= t.rows) {
        if (t.flags) {
            const uint2 f = *reinterpret_cast<const uint2 *>(t.flags + r);
            return nz_mask(f.x) | nz_mask(f.y) << 4;
        }
        const uint4 a = *reinterpret_cast<const uint4 *>(t.seen + r), b = *reinterpret_cast<const uint4 *>(t.seen + r + 4);
        return (uint32_t)(a.x != 0) | (uint32_t)(a.y != 0) << 1 | (uint32_t)(a.z != 0) << 2 | (uint32_t)(a.w != 0) << 3 |
               (uint32_t)(b.x != 0) << 4 | (uint32_t)(b.y != 0) << 5 | (uint32_t)(b.z != 0) << 6 | (uint32_t)(b.w != 0) << 7;
    }
    for (uint32_t k = 0; r + k < t.rows; k++) m |= (uint32_t)(t.flags ? t.flags[r + k] != 0 : t.seen[r + k] != 0) << k;
    return m;
}

// Sum over the block (valid in every thread); `part` is BLOCK / 64 words of LDS
__device__ __forceinline__ uint32_t block_sum(uint32_t v, uint32_t *part)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    uint32_t s = 0;
#pragma unroll
    for (int w = 0; w < BLOCK / 64; w++) s += part[w];
    return s;
}

__global__ void __launch_bounds__(BLOCK) k_sparse_count(SparseJobs jobs)
{
    __shared__ uint32_t part[BLOCK / 64];
    const int j = sparse_job(jobs);
    const uint32_t tile = blockIdx.x - jobs.first[j];
    const uint32_t c = block_sum(__popc(sparse_mask(jobs.t[j], tile * SPARSE_TILE + 8u * threadIdx.x)), part);
    if (threadIdx.x == 0) jobs.t[j].counts[tile] = c;
}

__global__ void __launch_bounds__(BLOCK) k_sparse_write(SparseJobs jobs)
{
    __shared__ uint32_t part[BLOCK / 64], wave_count[BLOCK / 64];
    __shared__ uint16_t list[SPARSE_TILE];
    const int j = sparse_job(jobs);
    const SparseTable &t = jobs.t[j];
    const uint32_t tile = blockIdx.x - jobs.first[j], t0 = tile * SPARSE_TILE;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t m = sparse_mask(t, t0 + 8u * threadIdx.x), before = 0;
    for (uint32_t i = threadIdx.x; i < tile; i += BLOCK) before += t.counts[i];
    const uint32_t base = block_sum(before, part);
    uint32_t total;
    uint32_t at = wave_prefix((uint32_t)__popc(m), lane, total);
    if (lane == 0) wave_count[wave] = total;
    __syncthreads();
    uint32_t count = 0;
#pragma unroll
    for (int w = 0; w < BLOCK / 64; w++) {
        if (w < wave) at += wave_count[w];
        count += wave_count[w];
    }
    for (; m; m &= m - 1) list[at++] = (uint16_t)(8u * threadIdx.x + (uint32_t)__builtin_ctz(m));
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < count; i += BLOCK) t.ids[base + i] = t0 + list[i];
    for (int c = 0; c < t.ncols; c++) {
        const bool wide = (t.is_u64 >> c) & 1u;
        for (uint32_t i = threadIdx.x; i < count; i += BLOCK) {
            const uint32_t r = t0 + list[i];
            const bool in = r < t.src_rows[c];
            if (wide) static_cast<uint64_t *>(t.dst[c])[base + i] = in ? static_cast<const uint64_t *>(t.src[c])[r] : 0ull;
            else static_cast<int32_t *>(t.dst[c])[base + i] = in ? static_cast<const int32_t *>(t.src[c])[r] : 0;
        }
    }
    if (threadIdx.x == 0 && t0 + SPARSE_TILE >= t.rows) *t.count = base + count;
}

// The statistics of compact probe tables (one block per table): the sum of
// the table's partial counts and its overflow flag, as the pair dst[2 y],
// dst[2 y + 1].
__global__ void __launch_bounds__(BLOCK) k_stats_reduce(StatsParts p, uint32_t *dst)
{
    __shared__ uint32_t wave_sum[BLOCK / 64];
    const int y = blockIdx.y;
    const uint32_t *st = p.stats[y];
    uint32_t t = 0;
    for (uint32_t i = threadIdx.x; i < p.nparts[y]; i += BLOCK) t += st[1 + i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) t += __shfl_down(t, off, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) wave_sum[wave] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t sum = 0;
#pragma unroll
        for (int w = 0; w < BLOCK / 64; w++) sum += wave_sum[w];
        dst[2 * y] = sum;
        dst[2 * y + 1] = st[0];
    }
}

__global__ void __launch_bounds__(BLOCK) k_gather_i32(const int32_t *src, const int32_t *ids, int64_t count,
                                                      int32_t *dst)
{
    for (int64_t j = (int64_t)blockIdx.x * BLOCK + threadIdx.x; j < count; j += (int64_t)gridDim.x * BLOCK)
        dst[j] = src[ids[j]];
}

__global__ void __launch_bounds__(BLOCK) k_minmax(const int32_t *col, int64_t n, int32_t *mm)
{
    int32_t lo = INT32_MAX, hi = INT32_MIN;
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK) {
        const int32_t v = col[i];
        lo = v < lo ? v : lo;
        hi = v > hi ? v : hi;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int32_t a = __shfl_xor(lo, off, 64), b = __shfl_xor(hi, off, 64);
        lo = a < lo ? a : lo;
        hi = b > hi ? b : hi;
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMin(&mm[0], lo);
        atomicMax(&mm[1], hi);
    }
}

__global__ void k_minmax_init(int32_t *mm)
{
    mm[0] = INT32_MAX;
    mm[1] = INT32_MIN;
}

// --------------------------------------------------------- dispatch helpers

void check_launch(const char *what)
{
    hip_check(hipGetLastError(), what);
}

unsigned grid_rows(int64_t n) { return stream_grid(n, ROWS_PER_STEP); }
unsigned grid_one(int64_t n) { return stream_grid(n, BLOCK); }

template <int CMP, int LOGIC>
void run_select_lit(const int32_t *col, const uint8_t *in, uint8_t *out, int64_t n, int32_t v, hipStream_t s)
{
    if (aligned(col, 16) && aligned(in, 4) && aligned(out, 4))
        hipLaunchKernelGGL((k_select_lit<CMP, LOGIC>), dim3(grid_rows(n)), dim3(BLOCK), 0, s, col, in, out, n, v);
    else
        hipLaunchKernelGGL((k_select_lit_row<CMP, LOGIC>), dim3(grid_one(n)), dim3(BLOCK), 0, s, col, in, out, n, v);
}

template <int CMP, int LOGIC>
void run_select_col(const int32_t *a, const int32_t *b, const uint8_t *in, uint8_t *out, int64_t n, hipStream_t s)
{
    if (aligned(a, 16) && aligned(b, 16) && aligned(in, 4) && aligned(out, 4))
        hipLaunchKernelGGL((k_select_col<CMP, LOGIC>), dim3(grid_rows(n)), dim3(BLOCK), 0, s, a, b, in, out, n);
    else
        hipLaunchKernelGGL((k_select_col_row<CMP, LOGIC>), dim3(grid_one(n)), dim3(BLOCK), 0, s, a, b, in, out, n);
}

template <int CMP>
void sel_lit_logic(int logic, const int32_t *col, const uint8_t *in, uint8_t *out, int64_t n, int32_t v, hipStream_t s)
{
    switch (logic) {
    case SDB_NONE: run_select_lit<CMP, SDB_NONE>(col, in, out, n, v, s); break;
    case SDB_AND: run_select_lit<CMP, SDB_AND>(col, in, out, n, v, s); break;
    default: run_select_lit<CMP, SDB_OR>(col, in, out, n, v, s); break;
    }
}

template <int CMP>
void sel_col_logic(int logic, const int32_t *a, const int32_t *b, const uint8_t *in, uint8_t *out, int64_t n, hipStream_t s)
{
    switch (logic) {
    case SDB_NONE: run_select_col<CMP, SDB_NONE>(a, b, in, out, n, s); break;
    case SDB_AND: run_select_col<CMP, SDB_AND>(a, b, in, out, n, s); break;
    default: run_select_col<CMP, SDB_OR>(a, b, in, out, n, s); break;
    }
}

template <int KIND>
void run_binop(int op, int32_t *r, const int32_t *a, const int32_t *b, int32_t lit, const uint8_t *f, int64_t n,
               hipStream_t s)
{
    const bool vec = aligned(r, 16) && aligned(f, 4) && (KIND == 1 || aligned(a, 16)) && (KIND == 2 || aligned(b, 16));
#define SDB_BINOP_CASE(OPV)                                                                              \
    case OPV:                                                                                            \
        if (vec)                                                                                         \
            hipLaunchKernelGGL((k_binop_vec<OPV, KIND>), dim3(grid_rows(n)), dim3(BLOCK), 0, s, r, a, b, lit, f, n); \
        else                                                                                             \
            hipLaunchKernelGGL((k_binop<OPV, KIND>), dim3(grid_one(n)), dim3(BLOCK), 0, s, r, a, b, lit, f, n); \
        break;
    switch (op) {
        SDB_BINOP_CASE(SDB_MUL)
        SDB_BINOP_CASE(SDB_DIV)
        SDB_BINOP_CASE(SDB_ADD)
        SDB_BINOP_CASE(SDB_SUB)
    }
#undef SDB_BINOP_CASE
}

} // namespace

// ------------------------------------------------------ internal launchers
// (used by the engine's unfused bundle path as well as the C ABI)

void launch_select_lit(const int32_t *col, const uint8_t *in, uint8_t *out, int64_t n, int cmp, int logic,
                       int32_t v, hipStream_t s)
{
    if (n <= 0) return;
    switch (cmp) {
    case SDB_EQ: sel_lit_logic<SDB_EQ>(logic, col, in, out, n, v, s); break;
    case SDB_NE: sel_lit_logic<SDB_NE>(logic, col, in, out, n, v, s); break;
    case SDB_LT: sel_lit_logic<SDB_LT>(logic, col, in, out, n, v, s); break;
    case SDB_LE: sel_lit_logic<SDB_LE>(logic, col, in, out, n, v, s); break;
    case SDB_GT: sel_lit_logic<SDB_GT>(logic, col, in, out, n, v, s); break;
    default: sel_lit_logic<SDB_GE>(logic, col, in, out, n, v, s); break;
    }
    check_launch("select_lit");
}

void launch_select_col(const int32_t *a, const int32_t *b, const uint8_t *in, uint8_t *out, int64_t n, int cmp,
                       int logic, hipStream_t s)
{
    if (n <= 0) return;
    switch (cmp) {
    case SDB_EQ: sel_col_logic<SDB_EQ>(logic, a, b, in, out, n, s); break;
    case SDB_NE: sel_col_logic<SDB_NE>(logic, a, b, in, out, n, s); break;
    case SDB_LT: sel_col_logic<SDB_LT>(logic, a, b, in, out, n, s); break;
    case SDB_LE: sel_col_logic<SDB_LE>(logic, a, b, in, out, n, s); break;
    case SDB_GT: sel_col_logic<SDB_GT>(logic, a, b, in, out, n, s); break;
    default: sel_col_logic<SDB_GE>(logic, a, b, in, out, n, s); break;
    }
    check_launch("select_col");
}

void launch_logical(const uint8_t *in, const uint8_t *local, uint8_t *out, int64_t n, int logic, hipStream_t s)
{
    if (n <= 0) return;
    if (aligned(in, 16) && aligned(local, 16) && aligned(out, 16)) {
        const unsigned grid = stream_grid((n >> 4) + 1, (int64_t)BLOCK * UNROLL);
        switch (logic) {
        case SDB_NONE: hipLaunchKernelGGL((k_logical_vec<SDB_NONE>), dim3(grid), dim3(BLOCK), 0, s, in, local, out, n); break;
        case SDB_AND: hipLaunchKernelGGL((k_logical_vec<SDB_AND>), dim3(grid), dim3(BLOCK), 0, s, in, local, out, n); break;
        default: hipLaunchKernelGGL((k_logical_vec<SDB_OR>), dim3(grid), dim3(BLOCK), 0, s, in, local, out, n); break;
        }
        check_launch("logical");
        return;
    }
    switch (logic) {
    case SDB_NONE: hipLaunchKernelGGL((k_logical<SDB_NONE>), dim3(grid_one(n)), dim3(BLOCK), 0, s, in, local, out, n); break;
    case SDB_AND: hipLaunchKernelGGL((k_logical<SDB_AND>), dim3(grid_one(n)), dim3(BLOCK), 0, s, in, local, out, n); break;
    default: hipLaunchKernelGGL((k_logical<SDB_OR>), dim3(grid_one(n)), dim3(BLOCK), 0, s, in, local, out, n); break;
    }
    check_launch("logical");
}

void launch_fill_i32(int32_t *dst, int32_t v, int64_t n, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fill_i32, dim3(stream_grid(n, BLOCK * 4)), dim3(BLOCK), 0, s, dst, v, n);
    check_launch("fill_i32");
}

void launch_fill_u8(uint8_t *dst, uint8_t v, int64_t n, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fill_u8, dim3(grid_one(std::max<int64_t>(n / 16, 1))), dim3(BLOCK), 0, s, dst, v, n);
    check_launch("fill_u8");
}

void launch_binop(int kind, int op, int32_t *r, const int32_t *a, const int32_t *b, int32_t lit,
                  const uint8_t *f, int64_t n, hipStream_t s)
{
    if (n <= 0) return;
    if (kind == 0) run_binop<0>(op, r, a, b, lit, f, n, s);
    else if (kind == 1) run_binop<1>(op, r, a, b, lit, f, n, s);
    else run_binop<2>(op, r, a, b, lit, f, n, s);
    check_launch("binop");
}

void launch_build_keys(const int32_t *keys, const uint8_t *flags, int64_t n, uint8_t *ht, int32_t len,
                       int32_t min, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_build_keys, dim3(grid_one(n)), dim3(BLOCK), 0, s, keys, flags, n, ht, len, min);
    check_launch("build_keys");
}

void launch_build_keyvals(const int32_t *keys, const int32_t *vals, const uint8_t *flags, int64_t n, int32_t *ht,
                          int32_t len, int32_t min, hipStream_t s)
{
    if (n <= 0) return;
    if (!aligned(ht, 8)) fail(SDB_ERR_INVALID_ARG, "key-value hash table must be 8-byte aligned");
    hipLaunchKernelGGL(k_build_keyvals, dim3(grid_one(n)), dim3(BLOCK), 0, s, keys, vals, flags, n, ht, len, min);
    check_launch("build_keyvals");
}

// A semi probe reads a bitmap in LDS where two blocks' bitmaps fit a CU and
// the column has 128 rows or more per table slot: every block reads the whole
// table first (16M rows, 300,000 slots: 21 us without, 26 with; 60M rows 78
// and 66; 6M rows, 20,000 slots 13 and 11).  A larger table would leave one
// block per CU (1.4M slots, 200M rows, 4 % flagged: 284 us without, 306 with).
// Where hardly a row is flagged the bitmap answers rows that nobody asks for
// (200M rows, 61,130 slots: none flagged 228 us without, 250 with; 0.5 % 238 and
// 252; 4 % 276 and 252; all 780 and 251); how many are is not known here.
constexpr int64_t SEMI_LDS_MIN_ROWS = 4 << 20;
constexpr int64_t SEMI_LDS_MIN_RATIO = 128;
constexpr int64_t SEMI_LDS_MAX_SLOTS = (int64_t)LDS_PER_CU / 2 * 8;

void launch_probe_semi(const int32_t *probe, const uint8_t *in, uint8_t *out, int64_t n, const uint8_t *ht,
                       int32_t min, int32_t max, hipStream_t s)
{
    if (n <= 0) return;
    const int vec = aligned(probe, 16) && aligned(in, 4) && aligned(out, 4);
    const int64_t len = max >= min ? (int64_t)max - min + 1 : 0;
    if (vec && aligned(ht, 16) && n >= SEMI_LDS_MIN_ROWS && len > 0 && len <= SEMI_LDS_MAX_SLOTS &&
        len * SEMI_LDS_MIN_RATIO <= n) {
        const size_t lds = ((size_t)len + 127) / 128 * 16;
        const dim3 grid(stream_grid(n, (int64_t)SEMI_BLOCK * UNROLL * 4, 2));
        hipLaunchKernelGGL(k_probe_semi_lds, grid, dim3(SEMI_BLOCK), lds, s, probe, in, out, n, ht, (uint32_t)len, min);
        check_launch("probe_semi");
        return;
    }
    hipLaunchKernelGGL(k_probe_semi, dim3(vec ? grid_rows(n) : grid_one(n)), dim3(BLOCK), 0, s, probe, in, out, n,
                       ht, min, max, vec);
    check_launch("probe_semi");
}

// a probe over at least this many rows, and at least this many rows per
// table slot, gathers from a 16-bit copy of a table of up to 2^26 slots
constexpr int64_t PROBE_U16_MIN_ROWS = 4 << 20;
constexpr int64_t PROBE_U16_MIN_RATIO = 16;
constexpr int64_t PROBE_U16_MAX_SLOTS = int64_t(1) << 26;

void launch_probe_full(const int32_t *probe, int32_t *val_out, const uint8_t *in, uint8_t *out, int64_t n,
                       const int32_t *ht, int32_t min, int32_t max, hipStream_t s)
{
    if (n <= 0) return;
    if (!aligned(ht, 8)) fail(SDB_ERR_INVALID_ARG, "key-value hash table must be 8-byte aligned");
    const int vec = aligned(probe, 16) && aligned(in, 4) && aligned(out, 4);
    PairsOrU16 t{reinterpret_cast<const int2 *>(ht), nullptr, nullptr};
    // a table much smaller than the probe column gets a 16-bit copy first
    // (two passes over the table; the probe then gathers 2 bytes per row
    // instead of 8)
    const int64_t len = max >= min ? (int64_t)max - min + 1 : 0;
    if (n >= PROBE_U16_MIN_ROWS && len > 0 && len * PROBE_U16_MIN_RATIO <= n && len <= PROBE_U16_MAX_SLOTS) {
        const size_t words = (size_t)((len + 31) / 32), part_off = 256;
        const size_t u16_off = part_off + PAIRS_RANGE_BLOCKS * 8, bits_off = u16_off + ((size_t)len * 2 + 15) / 16 * 16;
        const Scratch scratch(bits_off + words * 4, s);
        uint8_t *scr = scratch.data();
        int32_t *info = reinterpret_cast<int32_t *>(scr);
        int32_t *partials = reinterpret_cast<int32_t *>(scr + part_off);
        uint16_t *u16 = reinterpret_cast<uint16_t *>(scr + u16_off);
        uint32_t *bits = reinterpret_cast<uint32_t *>(scr + bits_off);
        const unsigned gr =
            (unsigned)std::min<int64_t>((len + BLOCK * UNROLL - 1) / (BLOCK * UNROLL), PAIRS_RANGE_BLOCKS);
        const unsigned g = (unsigned)std::min<int64_t>((len + BLOCK - 1) / BLOCK, 1024);
        hipLaunchKernelGGL(k_pairs_range, dim3(gr), dim3(BLOCK), 0, s, t.pairs, len, partials);
        hipLaunchKernelGGL(k_pairs_to_u16, dim3(g), dim3(BLOCK), 0, s, t.pairs, len, partials, (int)gr, info, u16, bits);
        t.u16 = u16;
        t.info = info;
        const dim3 grid(stream_grid(n, WT_ROWS * (PROBE_BLOCK / 64), 1));
        if (vec && len <= PROBE_LDS_SLOTS) {
            const size_t lds = ((size_t)len * 2 + 15) / 16 * 16;
            hipLaunchKernelGGL((k_probe_full_lds<true>), grid, dim3(PROBE_BLOCK), lds, s, probe, val_out, in, out, n, t,
                               bits, (uint32_t)words, 0u, 0u, min, max);
            check_launch("probe_full");
            return;
        }
        if (vec && len <= PROBE_FILTER_SLOTS) {
            uint32_t fwords = 1;
            while (fwords < words && fwords < PROBE_FILTER_WORDS) fwords *= 2;
            const uint32_t cap = probe_list_cap(fwords);
            const size_t lds = ((size_t)fwords + (PROBE_BLOCK / 64) * (64 + cap)) * 4;
            hipLaunchKernelGGL((k_probe_full_lds<false>), grid, dim3(PROBE_BLOCK), lds, s, probe, val_out, in, out, n, t,
                               bits, (uint32_t)words, fwords, cap, min, max);
            check_launch("probe_full");
            return;
        }
    }
    hipLaunchKernelGGL(k_probe_full, dim3(vec ? grid_rows(n) : grid_one(n)), dim3(BLOCK), 0, s, probe, val_out, in,
                       out, n, t, min, max, vec);
    check_launch("probe_full");
}

void launch_sum_flagged(const int32_t *col, const uint8_t *flags, int64_t n, uint64_t *acc, hipStream_t s)
{
    if (n <= 0) return;
    if (!aligned(acc, 8)) fail(SDB_ERR_INVALID_ARG, "accumulator must be 8-byte aligned");
    const int vec = aligned(col, 16) && aligned(flags, 4);
    const unsigned grid = stream_grid(n, (int64_t)RED_BLOCK * (vec ? 4 * UNROLL : 1), RED_PER_CU);
    hipLaunchKernelGGL(k_sum_flagged, dim3(grid), dim3(RED_BLOCK), 0, s, col, flags, n, acc, vec);
    check_launch("sum_flagged");
}

void launch_count_flags(const uint8_t *flags, int64_t n, uint64_t *out, bool accumulate, hipStream_t s)
{
    if (!aligned(out, 8)) fail(SDB_ERR_INVALID_ARG, "counter must be 8-byte aligned");
    if (!accumulate) {
        hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(1), 0, s, out);
        check_launch("count_flags init");
    }
    if (n <= 0) return;
    const unsigned grid = stream_grid(n, (int64_t)RED_BLOCK * 16 * UNROLL, RED_PER_CU);
    hipLaunchKernelGGL(k_count_flags, dim3(grid), dim3(RED_BLOCK), 0, s, flags, n, out);
    check_launch("count_flags");
}

// LDS budget of the privatised group-by (bytes); the slot array is u64 plus a
// one-bit occupancy map.
constexpr uint64_t GROUPBY_LDS_BYTES = 64 * 1024;

uint64_t groupby_lds_max_slots() { return (GROUPBY_LDS_BYTES * 8) / (64 + 1); }

void launch_groupby_dense(const int32_t *const *keys, int k, const int32_t *mins, const int32_t *maxs,
                          const int32_t *agg, const uint8_t *flags, int64_t n, int32_t *const *out_keys,
                          uint64_t *sums, uint32_t *seen, uint64_t prod, hipStream_t s, int strategy)
{
    if (k < 1 || k > GB_MAX_KEYS) fail(SDB_ERR_INVALID_ARG, "group-by supports 1..8 key columns");
    if (prod == 0) fail(SDB_ERR_INVALID_ARG, "group-by range product is 0");
    if (n <= 0) return;
    GroupArgs g{};
    g.k = k;
    for (int j = 0; j < k; j++) {
        g.keys[j] = keys[j];
        g.out_keys[j] = out_keys[j];
        g.mins[j] = mins[j];
        g.maxs[j] = maxs[j];
        g.range[j] = (uint32_t)maxs[j] - (uint32_t)mins[j] + 1u;
    }
    // the slot decode at flush is exact when the in-range index cannot wrap
    uint64_t exact = 1;
    bool fits = true;
    for (int j = 0; j < k; j++) {
        if (maxs[j] < mins[j]) fits = false;
        exact *= (uint64_t)((int64_t)maxs[j] - (int64_t)mins[j] + 1);
        if (exact > prod) fits = false;
    }
    fits = fits && exact == prod;
    const bool lds = strategy != 1 && fits && prod <= groupby_lds_max_slots();
    if (lds) {
        // 1024-thread blocks share one LDS copy of the sums among 16 waves;
        // as many blocks per CU as that LDS allows (at most 2)
        const size_t bytes = prod * 8 + ((prod + 31) / 32) * 4;
        const size_t used = bytes + (GB_BLOCK / 64) * GB_LIST * sizeof(uint16_t);
        const int per_cu = std::max(1, std::min(2, (int)(LDS_PER_CU / used)));
        const dim3 grid(stream_grid(n, WT_ROWS * (GB_BLOCK / 64), per_cu));
#define SDB_GROUPBY_CASE(KV)                                                                                     \
    hipLaunchKernelGGL((k_groupby_lds<KV>), grid, dim3(GB_BLOCK), bytes, s, g, agg, flags, n, sums, seen,        \
                       (uint32_t)prod);                                                                          \
    break;
        switch (k) {
        case 1: SDB_GROUPBY_CASE(1)
        case 2: SDB_GROUPBY_CASE(2)
        case 3: SDB_GROUPBY_CASE(3)
        case 4: SDB_GROUPBY_CASE(4)
        default: SDB_GROUPBY_CASE(0)
        }
#undef SDB_GROUPBY_CASE
    } else {
        hipLaunchKernelGGL(k_groupby_global, dim3(grid_one(n)), dim3(BLOCK), 0, s, g, agg, flags, n, sums, seen,
                           prod);
    }
    check_launch("groupby_dense");
}

void launch_seen_to_flags(const uint32_t *seen, uint8_t *flags, uint64_t prod, hipStream_t s)
{
    if (prod == 0) return;
    hipLaunchKernelGGL(k_seen_to_flags, dim3(grid_one((int64_t)prod)), dim3(BLOCK), 0, s, seen, flags, prod);
    check_launch("seen_to_flags");
}

uint32_t bits_partials(int32_t len)
{
    if (len <= 0) return 0;
    const int64_t per_block = 64 * BITS_GROUPS * (BLOCK / 64);
    return (uint32_t)std::min<int64_t>(BITS_MAX_BLOCKS, ((int64_t)len + per_block - 1) / per_block);
}

template <int N> static int launch_tables(const CompactJob *jobs, int n, hipStream_t s)
{
    BitsJobs<N> bj{};
    RankJobs<N> rj{};
    std::fill(std::begin(bj.first), std::end(bj.first), UINT32_MAX);
    std::fill(std::begin(rj.first), std::end(rj.first), UINT32_MAX);
    uint32_t blocks = 0, ranges = 0;
    int nbits = 0, nrank = 0;
    for (int i = 0; i < n; i++) {
        const CompactJob &c = jobs[i];
        if (c.len <= 0) continue;
        if (c.pairs && !aligned(c.ht, 8)) fail(SDB_ERR_INVALID_ARG, "key-value hash table must be 8-byte aligned");
        const uint32_t nblocks = bits_partials(c.len);
        bj.first[nbits] = blocks;
        bj.job[nbits++] = {c.ht, c.bits, c.vals, c.partials, c.bad, c.len, c.vmin, nblocks, c.pairs ? 1u : 0u};
        blocks += nblocks;
        if (!c.dict) continue;
        const uint32_t words = (uint32_t)(((int64_t)c.len + 31) / 32);
        if (c.dict_cap < rank_values_off(words)) fail(SDB_ERR_RUNTIME, "rank dictionary buffer too small");
        // the bitmap kernel's blocks each counted one run of 32 words when
        // the job's blocks cover the table without wrapping (below 2^21
        // slots; dictionaries are built for tables far smaller)
        static_assert(64 * BITS_GROUPS * (BLOCK / 64) == 32 * RANK_PART_WORDS, "one bitmap block per 32 words");
        const uint32_t r = (words + RANK_PART_WORDS - 1) / RANK_PART_WORDS;
        if (!c.partials || !c.vals || r != nblocks)
            fail(SDB_ERR_RUNTIME, "rank dictionary: the bitmap's per-block counts do not cover 32 words each");
        rj.first[nrank] = ranges;
        rj.job[nrank++] = {c.bits, c.partials, c.vals, c.dict, c.len, (int32_t)words,
                           (c.dict_cap - rank_values_off(words)) / 2u};
        ranges += r;
    }
    if (nbits) {
        hipLaunchKernelGGL((k_compact_bits<N>), dim3(blocks), dim3(BLOCK), 0, s, bj);
        check_launch("compact_bits");
    }
    if (nrank) {
        hipLaunchKernelGGL((k_rank_dicts<N>), dim3(ranges), dim3(64), 0, s, rj);
        check_launch("rank_dicts");
    }
    return (nbits ? 1 : 0) + (nrank ? 1 : 0);
}

int launch_compact_tables(const CompactJob *jobs, size_t njobs, hipStream_t s)
{
    int launches = 0;
    for (size_t at = 0; at < njobs; at += COMPACT_JOBS) {
        const int n = (int)std::min<size_t>(COMPACT_JOBS, njobs - at);
        launches += n <= COMPACT_JOBS_SMALL ? launch_tables<COMPACT_JOBS_SMALL>(jobs + at, n, s)
                                            : launch_tables<COMPACT_JOBS>(jobs + at, n, s);
    }
    return launches;
}

void launch_stats_reduce(const StatsParts &p, uint32_t *dst, hipStream_t s)
{
    if (p.n <= 0) return;
    if (p.n > PACK_MAX_PARTS) fail(SDB_ERR_INVALID_ARG, "stats reduce: too many tables");
    hipLaunchKernelGGL(k_stats_reduce, dim3(1, (unsigned)p.n), dim3(BLOCK), 0, s, p, dst);
    check_launch("stats_reduce");
}

void launch_batch_masks(const FMaskCol *cols, const uint32_t *lens, int ncols, const FMaskEntry *ents, hipStream_t s)
{
    if (ncols <= 0) return;
    if (ncols > F_MASK_MAX_COLS) fail(SDB_ERR_RUNTIME, "batch masks: too many columns");
    MaskGrid grid;
    std::fill(std::begin(grid.first), std::end(grid.first), UINT32_MAX);
    uint32_t blocks = 0;
    for (int c = 0; c < ncols; c++) {
        grid.first[c] = blocks;
        blocks += (lens[c] + MASK_KEYS - 1) / MASK_KEYS;
    }
    if (!blocks) return;
    hipLaunchKernelGGL(k_batch_masks, dim3(blocks), dim3(BLOCK), 0, s, cols, ents, grid);
    check_launch("batch_masks");
}

void launch_batch_dict(const FMaskDict *dicts, int ndicts, hipStream_t s)
{
    if (ndicts <= 0) return;
    hipLaunchKernelGGL(k_batch_dict, dim3((unsigned)ndicts), dim3(DICT_BLOCK), 0, s, dicts);
    check_launch("batch_dict");
}

int64_t compact_tiles(int64_t n) { return n > 0 ? (n + COMPACT_TILE - 1) / COMPACT_TILE : 0; }

void launch_compact(const uint8_t *flags, int64_t n, int32_t *row_ids, uint32_t *count, hipStream_t s)
{
    const int64_t ntiles = compact_tiles(n);
    const Scratch scratch((size_t)std::max<int64_t>(ntiles, 1) * 4, s);
    launch_compact_into(flags, n, row_ids, count, reinterpret_cast<uint32_t *>(scratch.data()), s);
}

void launch_compact_into(const uint8_t *flags, int64_t n, int32_t *row_ids, uint32_t *count, uint32_t *counts,
                         hipStream_t s)
{
    const int64_t ntiles = compact_tiles(n);
    const dim3 grid((unsigned)((ntiles + COMPACT_WAVES - 1) / COMPACT_WAVES));
    if (ntiles > 0) hipLaunchKernelGGL(k_compact_count, grid, dim3(BLOCK), 0, s, flags, n, ntiles, counts);
    hipLaunchKernelGGL(k_compact_scan, dim3(1), dim3(SCAN_BLOCK), 0, s, counts, ntiles, count);
    if (ntiles > 0)
        hipLaunchKernelGGL(k_compact_write, grid, dim3(BLOCK), 0, s, flags, n, ntiles, counts, row_ids);
    check_launch("compact");
}

// ------------------------------------------- compaction without allocation
//
// The per-tile counts of sdb_compact_noalloc live in a fixed device array of
// the library instead of library-allocated scratch: each GPU the library runs
// on holds its own copy until the process ends.  Host code never passes the
// array's name to a kernel (on the host it only stands for the symbol); its
// device address is looked up once per device, with that device current, by
// hipGetSymbolAddress, and that address is what the kernels get.  Every call
// on one GPU shares the array; the counting pass overwrites every count the
// scan and write passes read, so nothing needs clearing between calls.
constexpr int64_t NOALLOC_TILES = 65536; // 256 KiB of counts: 2^28 rows
static_assert(NOALLOC_TILES * COMPACT_TILE == (int64_t(1) << 28), "noalloc compaction covers 2^28 rows");
static __device__ __align__(256) uint32_t scratch[NOALLOC_TILES];
constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex g_noalloc_mu;
uint32_t *g_noalloc_ptr[NOALLOC_MAX_DEVICES] = {};

uint32_t *noalloc_counts()
{
    int dev = 0;
    SDB_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) fail(SDB_ERR_UNSUPPORTED, "device ordinal beyond the no-allocation table");
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
        void *ptr = nullptr;
        hip_check(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
        if (!ptr) fail(SDB_ERR_HIP, "hipGetSymbolAddress(scratch) returned null");
        g_noalloc_ptr[dev] = static_cast<uint32_t *>(ptr);
    }
    return g_noalloc_ptr[dev];
}

void launch_compact_noalloc(const uint8_t *flags, int64_t n, int32_t *row_ids, uint32_t *count, hipStream_t s)
{
    if (n > NOALLOC_TILES * COMPACT_TILE)
        fail(SDB_ERR_INVALID_ARG, "sdb_compact_noalloc: n exceeds 2^28 rows (the fixed tile-count array)");
    launch_compact_into(flags, n, row_ids, count, noalloc_counts(), s);
}

void launch_gather_cols(const GatherCols &g, const int32_t *ids, int64_t count, hipStream_t s)
{
    if (count <= 0 || g.ncols <= 0) return;
    if (g.ncols > GATHER_MAX_COLS) fail(SDB_ERR_INVALID_ARG, "gather: too many columns");
    hipLaunchKernelGGL(k_gather_cols, dim3(grid_one(count)), dim3(BLOCK), 0, s, g, ids, count);
    check_launch("gather_cols");
}

void launch_pack_parts(const PackParts &p, uint8_t *dst, hipStream_t s)
{
    if (p.n <= 0) return;
    if (p.n > PACK_MAX_PARTS) fail(SDB_ERR_INVALID_ARG, "pack: too many parts");
    uint64_t most = 0;
    for (int i = 0; i < p.n; i++) most = std::max(most, p.bytes[i]);
    const unsigned gx = (unsigned)std::max<uint64_t>(1, std::min<uint64_t>((most / 16 + BLOCK - 1) / BLOCK, 256));
    auto launch = [&](auto list) {
        for (int i = 0; i < p.n; i++) {
            list.src[i] = p.src[i];
            list.off[i] = p.off[i];
            list.bytes[i] = p.bytes[i];
            list.kind[i] = p.kind[i];
        }
        constexpr int N = sizeof(list.kind);
        hipLaunchKernelGGL((k_pack_parts<N>), dim3(gx, (unsigned)p.n), dim3(BLOCK), 0, s, list, dst);
    };
    if (p.n <= PACK_FEW) launch(PackList<PACK_FEW>{});
    else launch(PackList<PACK_MAX_PARTS>{});
    check_launch("pack_parts");
}

uint64_t sparse_tiles(uint64_t rows) { return (rows + SPARSE_TILE - 1) / SPARSE_TILE; }

int launch_sparse_tables(const SparseTable *t, size_t n, hipStream_t s)
{
    int launches = 0;
    for (size_t at = 0; at < n; at += SPARSE_TABLES) {
        SparseJobs jobs{};
        std::fill(std::begin(jobs.first), std::end(jobs.first), UINT32_MAX);
        uint32_t blocks = 0;
        for (size_t i = 0; i < (size_t)SPARSE_TABLES && at + i < n; i++) {
            const SparseTable &T = t[at + i];
            if (T.rows == 0 || T.rows > SPARSE_MAX_ROWS || T.ncols > GATHER_MAX_COLS || (!T.flags && !T.seen) ||
                !aligned(T.flags, 8) || !aligned(T.seen, 16))
                fail(SDB_ERR_RUNTIME, "sparse result table out of the kernels' range");
            jobs.first[i] = blocks;
            jobs.t[i] = T;
            blocks += (uint32_t)sparse_tiles(T.rows);
        }
        if (!blocks) continue;
        hipLaunchKernelGGL(k_sparse_count, dim3(blocks), dim3(BLOCK), 0, s, jobs);
        hipLaunchKernelGGL(k_sparse_write, dim3(blocks), dim3(BLOCK), 0, s, jobs);
        check_launch("sparse_tables");
        launches += 2;
    }
    return launches;
}

void launch_gather_i32(const int32_t *src, const int32_t *ids, int64_t count, int32_t *dst, hipStream_t s)
{
    if (count <= 0) return;
    hipLaunchKernelGGL(k_gather_i32, dim3(grid_one(count)), dim3(BLOCK), 0, s, src, ids, count, dst);
    check_launch("gather_i32");
}

void minmax_i32(const int32_t *col, int64_t n, int32_t *mn, int32_t *mx, hipStream_t s)
{
    if (n <= 0) fail(SDB_ERR_INVALID_ARG, "min/max of an empty column");
    const Scratch scratch(8, s);
    int32_t *mm = reinterpret_cast<int32_t *>(scratch.data());
    hipLaunchKernelGGL(k_minmax_init, dim3(1), dim3(1), 0, s, mm);
    hipLaunchKernelGGL(k_minmax, dim3(grid_one(n)), dim3(BLOCK), 0, s, col, n, mm);
    check_launch("minmax");
    int32_t host[2];
    SDB_HIP(hipMemcpyAsync(host, mm, 8, hipMemcpyDeviceToHost, s));
    SDB_HIP(hipStreamSynchronize(s));
    *mn = host[0];
    *mx = host[1];
}

} // namespace sdb

// =================================================================== C ABI

using namespace sdb;

namespace {
inline void check_n(int64_t n) { require(n >= 0, "negative length"); }
inline void check_cmp(int cmp) { require(cmp >= SDB_EQ && cmp <= SDB_GE, "comparison op out of range"); }
inline void check_logic(int l) { require(l >= SDB_NONE && l <= SDB_OR, "logical op out of range"); }
inline void check_binop(int op) { require(op >= SDB_MUL && op <= SDB_SUB, "arithmetic op out of range"); }
} // namespace

extern "C" {

int sdb_comp_op_from_string(const char *op)
{
    const std::string s = op ? op : "";
    if (s == "==") return SDB_EQ;
    if (s == ">=") return SDB_GE;
    if (s == "<=") return SDB_LE;
    if (s == "<") return SDB_LT;
    if (s == ">") return SDB_GT;
    if (s == "!=" || s == "<>") return SDB_NE;
    return SDB_EQ;
}

int sdb_logical_op_from_string(const char *op)
{
    const std::string s = op ? op : "";
    if (s == "AND") return SDB_AND;
    if (s == "OR") return SDB_OR;
    return SDB_NONE;
}

int sdb_binop_from_string(const char *op)
{
    const std::string s = op ? op : "";
    if (s == "*") return SDB_MUL;
    if (s == "/") return SDB_DIV;
    if (s == "+") return SDB_ADD;
    if (s == "-") return SDB_SUB;
    return -1;
}

int sdb_select_lit(const int32_t *col, const uint8_t *in_flags, uint8_t *out_flags, int64_t n, int cmp, int logic,
                   int32_t value, sdb_stream stream)
{
    return guarded([&] {
        check_n(n), check_cmp(cmp), check_logic(logic);
        require(n == 0 || (col && in_flags && out_flags), "null pointer");
        launch_select_lit(col, in_flags, out_flags, n, cmp, logic, value, as_stream(stream));
    });
}

int sdb_select_col(const int32_t *a, const int32_t *b, const uint8_t *in_flags, uint8_t *out_flags, int64_t n,
                   int cmp, int logic, sdb_stream stream)
{
    return guarded([&] {
        check_n(n), check_cmp(cmp), check_logic(logic);
        require(n == 0 || (a && b && in_flags && out_flags), "null pointer");
        launch_select_col(a, b, in_flags, out_flags, n, cmp, logic, as_stream(stream));
    });
}

int sdb_logical(const uint8_t *in_flags, const uint8_t *local_flags, uint8_t *out_flags, int64_t n, int logic,
                sdb_stream stream)
{
    return guarded([&] {
        check_n(n), check_logic(logic);
        require(n == 0 || (in_flags && local_flags && out_flags), "null pointer");
        launch_logical(in_flags, local_flags, out_flags, n, logic, as_stream(stream));
    });
}

int sdb_fill_i32(int32_t *dst, int32_t value, int64_t n, sdb_stream stream)
{
    return guarded([&] {
        check_n(n);
        require(n == 0 || dst, "null pointer");
        require(((uintptr_t)dst & 3) == 0, "int32 column must be 4-byte aligned");
        launch_fill_i32(dst, value, n, as_stream(stream));
    });
}

int sdb_binop_cc(int32_t *result, const int32_t *a, const int32_t *b, const uint8_t *flags, int64_t n, int op,
                 sdb_stream stream)
{
    return guarded([&] {
        check_n(n), check_binop(op);
        require(n == 0 || (result && a && b && flags), "null pointer");
        launch_binop(0, op, result, a, b, 0, flags, n, as_stream(stream));
    });
}

int sdb_binop_lc(int32_t *result, int32_t a, const int32_t *b, const uint8_t *flags, int64_t n, int op,
                 sdb_stream stream)
{
    return guarded([&] {
        check_n(n), check_binop(op);
        require(n == 0 || (result && b && flags), "null pointer");
        launch_binop(1, op, result, nullptr, b, a, flags, n, as_stream(stream));
    });
}

int sdb_binop_cl(int32_t *result, const int32_t *a, int32_t b, const uint8_t *flags, int64_t n, int op,
                 sdb_stream stream)
{
    return guarded([&] {
        check_n(n), check_binop(op);
        require(n == 0 || (result && a && flags), "null pointer");
        launch_binop(2, op, result, a, nullptr, b, flags, n, as_stream(stream));
    });
}

int sdb_build_keys(const int32_t *keys, const uint8_t *flags, int64_t n, uint8_t *ht, int32_t ht_len,
                   int32_t ht_min, sdb_stream stream)
{
    return guarded([&] {
        check_n(n);
        require(ht_len > 0, "hash table length must be positive");
        require(n == 0 || (keys && flags && ht), "null pointer");
        launch_build_keys(keys, flags, n, ht, ht_len, ht_min, as_stream(stream));
    });
}

int sdb_build_keyvals(const int32_t *keys, const int32_t *vals, const uint8_t *flags, int64_t n, int32_t *ht,
                      int32_t ht_len, int32_t ht_min, sdb_stream stream)
{
    return guarded([&] {
        check_n(n);
        require(ht_len > 0, "hash table length must be positive");
        require(n == 0 || (keys && vals && flags && ht), "null pointer");
        launch_build_keyvals(keys, vals, flags, n, ht, ht_len, ht_min, as_stream(stream));
    });
}

int sdb_probe_semi(const int32_t *probe, const uint8_t *in_flags, uint8_t *out_flags, int64_t n, const uint8_t *ht,
                   int32_t ht_min, int32_t ht_max, sdb_stream stream)
{
    return guarded([&] {
        check_n(n);
        require(ht_max >= ht_min, "ht_max < ht_min");
        require(n == 0 || (probe && in_flags && out_flags && ht), "null pointer");
        launch_probe_semi(probe, in_flags, out_flags, n, ht, ht_min, ht_max, as_stream(stream));
    });
}

int sdb_probe_full(const int32_t *probe, int32_t *val_out, const uint8_t *in_flags, uint8_t *out_flags, int64_t n,
                   const int32_t *ht, int32_t ht_min, int32_t ht_max, sdb_stream stream)
{
    return guarded([&] {
        check_n(n);
        require(ht_max >= ht_min, "ht_max < ht_min");
        require(n == 0 || (probe && val_out && in_flags && out_flags && ht), "null pointer");
        launch_probe_full(probe, val_out, in_flags, out_flags, n, ht, ht_min, ht_max, as_stream(stream));
    });
}

int sdb_sum_flagged(const int32_t *col, const uint8_t *flags, int64_t n, uint64_t *acc, sdb_stream stream)
{
    return guarded([&] {
        check_n(n);
        require(acc, "null accumulator");
        require(n == 0 || (col && flags), "null pointer");
        launch_sum_flagged(col, flags, n, acc, as_stream(stream));
    });
}

int sdb_groupby_dense(const int32_t *const *keys, int k, const int32_t *mins, const int32_t *maxs,
                      const int32_t *agg, const uint8_t *flags, int64_t n, int32_t *const *out_keys,
                      uint64_t *sums, uint32_t *seen, uint64_t prod, sdb_stream stream)
{
    return guarded([&] {
        check_n(n);
        require(keys && mins && maxs && out_keys, "null pointer");
        require(prod == 0 || (sums && seen), "null pointer");
        require(n == 0 || (agg && flags), "null pointer");
        for (int j = 0; j < k && j < 8; j++) require(n == 0 || (keys[j] && out_keys[j]), "null key column");
        launch_groupby_dense(keys, k, mins, maxs, agg, flags, n, out_keys, sums, seen, prod, as_stream(stream), 0);
    });
}

int sdb_seen_to_flags(const uint32_t *seen, uint8_t *flags, uint64_t prod, sdb_stream stream)
{
    return guarded([&] {
        require(prod == 0 || (seen && flags), "null pointer");
        launch_seen_to_flags(seen, flags, prod, as_stream(stream));
    });
}

int sdb_count_flags(const uint8_t *flags, int64_t n, uint64_t *out, int accumulate, sdb_stream stream)
{
    return guarded([&] {
        check_n(n);
        require(out, "null output");
        require(n == 0 || flags, "null pointer");
        launch_count_flags(flags, n, out, accumulate != 0, as_stream(stream));
    });
}

int sdb_compact(const uint8_t *flags, int64_t n, int32_t *row_ids, uint32_t *count, sdb_stream stream)
{
    return guarded([&] {
        check_n(n);
        require(n <= INT32_MAX, "compaction is limited to 2^31-1 rows (int32 row ids)");
        require(count, "null count");
        require(n == 0 || (flags && row_ids), "null pointer");
        launch_compact(flags, n, row_ids, count, as_stream(stream));
    });
}

int sdb_compact_noalloc(const uint8_t *flags, int64_t n, int32_t *row_ids, uint32_t *count, sdb_stream stream)
{
    return guarded([&] {
        check_n(n);
        require(n <= SDB_COMPACT_NOALLOC_MAX_ROWS, "sdb_compact_noalloc: n exceeds SDB_COMPACT_NOALLOC_MAX_ROWS (2^28)");
        require(count, "null count");
        require(n == 0 || (flags && row_ids), "null pointer");
        launch_compact_noalloc(flags, n, row_ids, count, as_stream(stream));
    });
}

int sdb_gather_i32(const int32_t *src, const int32_t *row_ids, int64_t count, int32_t *dst, sdb_stream stream)
{
    return guarded([&] {
        check_n(count);
        require(count == 0 || (src && row_ids && dst), "null pointer");
        launch_gather_i32(src, row_ids, count, dst, as_stream(stream));
    });
}

int sdb_compress_sync(const int32_t *const *cols, int ncols, const uint8_t *flags, int64_t n,
                      int32_t *const *host_cols, uint64_t *count, sdb_stream stream)
{
    return guarded([&] {
        check_n(n);
        require(n <= INT32_MAX, "compress_sync is limited to 2^31-1 rows (int32 row ids)");
        require(ncols >= 0 && ncols <= GATHER_MAX_COLS, "compress_sync: 0 to 8 columns");
        require(count && (ncols == 0 || (cols && host_cols)), "null pointer");
        *count = 0;
        if (n == 0) return;
        for (int c = 0; c < ncols; c++) require(cols[c] && host_cols[c], "null column");
        require(flags, "null flags");
        hipStream_t s = as_stream(stream);
        // device half: the selected rows' ids (build_row_ids,
        // models/transient_table.hpp:535-599, here in row order) ...
        const int64_t ntiles = compact_tiles(n);
        const size_t ids_bytes = ((size_t)n * 4 + 255) / 256 * 256, cnt_off = ids_bytes + (size_t)ntiles * 4;
        const Scratch scratch(cnt_off + 256, s);
        uint8_t *scr = scratch.data();
        int32_t *ids = reinterpret_cast<int32_t *>(scr);
        uint32_t *dcount = reinterpret_cast<uint32_t *>(scr + cnt_off);
        launch_compact_into(flags, n, ids, dcount, reinterpret_cast<uint32_t *>(scr + ids_bytes), s);
        uint32_t selected = 0;
        SDB_HIP(hipMemcpyAsync(&selected, dcount, 4, hipMemcpyDeviceToHost, s));
        SDB_HIP(hipStreamSynchronize(s));
        *count = selected;
        if (selected == 0 || ncols == 0) return;
        // ... and their values, gathered (Segment::compress_sync,
        // models/models.hpp:1019-1035) and copied to the host with the ids
        int32_t *vals = nullptr;
        SDB_HIP(hipMalloc(&vals, (size_t)selected * 4 * (size_t)ncols));
        std::vector<int32_t> hids(selected), hvals((size_t)selected * (size_t)ncols);
        hipError_t e = hipSuccess;
        try {
            GatherCols g{};
            for (int c = 0; c < ncols; c++) {
                g.src[c] = cols[c];
                g.dst[c] = vals + (size_t)c * selected;
                g.src_rows[c] = (uint64_t)n;
            }
            g.ncols = ncols;
            launch_gather_cols(g, ids, selected, s);
            e = hipMemcpyAsync(hids.data(), ids, (size_t)selected * 4, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess)
                e = hipMemcpyAsync(hvals.data(), vals, hvals.size() * 4, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipStreamSynchronize(s);
        } catch (...) {
            (void)hipStreamSynchronize(s);
            (void)hipFree(vals);
            throw;
        }
        (void)hipFree(vals);
        hip_check(e, "compress_sync copy");
        // host half: the scatter into the host columns (models.hpp:1044-1063)
        for (int c = 0; c < ncols; c++) {
            const int32_t *v = hvals.data() + (size_t)c * selected;
            int32_t *dst = host_cols[c];
            for (uint32_t j = 0; j < selected; j++) dst[hids[j]] = v[j];
        }
    });
}

int sdb_minmax_i32(const int32_t *col, int64_t n, int32_t *min_out, int32_t *max_out, sdb_stream stream)
{
    return guarded([&] {
        require(n > 0, "min/max needs at least one row");
        require(col && min_out && max_out, "null pointer");
        minmax_i32(col, n, min_out, max_out, as_stream(stream));
    });
}

} // extern "C"
