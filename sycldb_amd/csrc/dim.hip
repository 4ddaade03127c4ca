// The build sides of a plan's joins: filter a dimension table and insert its
// keys (and values) into the reference-layout hash table, for several tables
// in one launch.
//
// Each is a short fused program over 2,556 to a few million rows.  As one
// launch per table they cost the host 4 to 8 us each and the device 4 to 11 us
// each, one after another: most of a small query, and of a batch's start.  The
// programs of one plan or batch do not read each other's output, so they are
// queued and run side by side: block b works on the job whose blocks
// [first[j], first[j + 1]) hold it, 1,024 rows per block and step, and runs
// the job's program from the kernel arguments (uniform, so every dispatch is a
// scalar branch).
#include "capi_util.hpp"
#include "fused.hpp"
#include "fused_device.hpp"

#include <algorithm>

namespace sdb {

namespace {

constexpr int DIM_BLOCK = 256;
constexpr int64_t DIM_STEP = 4 * DIM_BLOCK; // rows per block and step
constexpr int64_t DIM_MAX_BLOCKS = 1024;    // per job

// A plan has at most four joins in most schemas: its launch takes the small
// form, whose arguments are a fifth of the large one's (3 KB of arguments cost
// the host about 2 us a launch more than 0.6 KB).
constexpr int DIM_JOBS_SMALL = 4;
template <int N> struct DimJobs {
    uint32_t first[N]; // first block of each job (unused: UINT32_MAX)
    uint32_t nblocks[N];
    DimJob job[N];
};
static_assert(sizeof(DimJobs<DIM_JOBS>) <= 4096, "kernel argument segment");

// rows r .. r + 3 of a column (rows at or past n: 0)
__device__ __forceinline__ int4 dim_rows(const int32_t *col, int64_t r, int64_t n, bool vec)
{
    if (vec && r + 4 <= n) return *reinterpret_cast<const int4 *>(col + r);
    int32_t x[4];
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = r + k < n ? col[r + k] : 0;
    return make_int4(x[0], x[1], x[2], x[3]);
}

template <int N> __global__ void __launch_bounds__(DIM_BLOCK) k_dim_builds(DimJobs<N> jobs)
{
    int j = 0;
#pragma unroll
    for (int k = 1; k < N; k++) j += blockIdx.x >= jobs.first[k];
    const DimJob &J = jobs.job[j];
    const int64_t n = J.n, stride = (int64_t)jobs.nblocks[j] * DIM_STEP;
    const bool vec = J.vec != 0;
    for (int64_t r = (int64_t)(blockIdx.x - jobs.first[j]) * DIM_STEP + 4 * threadIdx.x; r < n; r += stride) {
        const int4 zero = make_int4(0, 0, 0, 0);
        const int4 c0 = dim_rows(J.col[0], r, n, vec);
        const int4 c1 = J.ncols > 1 ? dim_rows(J.col[1], r, n, vec) : zero;
        const int4 c2 = J.ncols > 2 ? dim_rows(J.col[2], r, n, vec) : zero;
        const int4 c3 = J.ncols > 3 ? dim_rows(J.col[3], r, n, vec) : zero;
        auto column = [&](int c) { return c == 0 ? c0 : c == 1 ? c1 : c == 2 ? c2 : c3; };
        uint32_t F = J.init; // flag register f of row k: bit 4 f + k
        for (int i = 0; i < J.ninstr; i++) {
            const DimInstr &I = J.ins[i];
            const uint32_t in = (F >> (4 * I.fin)) & 15u;
            uint32_t p = 0;
            if (I.kind == FK_LOGICAL) {
                p = (F >> (4 * I.floc)) & 15u;
            } else {
                const int4 x = column(I.a);
                const int32_t xs[4] = {x.x, x.y, x.z, x.w};
                if (I.kind == FK_SEL_LIT) {
#pragma unroll
                    for (int k = 0; k < 4; k++) p |= (uint32_t)compare(I.cmp, xs[k], I.lit) << k;
                } else if (I.kind == FK_SEL_RANGE) {
#pragma unroll
                    for (int k = 0; k < 4; k++) p |= (uint32_t)(xs[k] >= I.lit && xs[k] <= I.lit2) << k;
                } else if (I.kind == FK_SEL_IN2) {
#pragma unroll
                    for (int k = 0; k < 4; k++) p |= (uint32_t)(xs[k] == I.lit || xs[k] == I.lit2) << k;
                } else { // FK_SEL_COL
                    const int4 y = column(I.b);
                    const int32_t ys[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
                    for (int k = 0; k < 4; k++) p |= (uint32_t)compare(I.cmp, xs[k], ys[k]) << k;
                }
            }
            const uint32_t out = I.logic == SDB_NONE ? p : I.logic == SDB_AND ? (in & p) : (in | p);
            F = (F & ~(15u << (4 * I.fout))) | out << (4 * I.fout);
        }
        if (J.store) {
            const uint32_t m = (F >> (4 * J.store_reg)) & 15u, w = (m * 0x00204081u) & 0x01010101u;
            if (vec && r + 4 <= n) *reinterpret_cast<uint32_t *>(J.store + r) = w;
            else
                for (int k = 0; k < 4; k++)
                    if (r + k < n) J.store[r + k] = (uint8_t)(w >> (8 * k));
        }
        const uint32_t in = (F >> (4 * J.fin)) & 15u;
        const int4 key = column(J.key), val = column(J.val);
        const int32_t keys[4] = {key.x, key.y, key.z, key.w}, vals[4] = {val.x, val.y, val.z, val.w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t s = slot_of(keys[k], J.ht_min);
            if (r + k >= n || s >= (uint32_t)J.ht_len) continue;
            if (!J.pairs) static_cast<uint8_t *>(J.ht)[s] = (in >> k) & 1u;
            else if ((in >> k) & 1u) static_cast<int2 *>(J.ht)[s] = make_int2(1, vals[k]);
            else static_cast<int32_t *>(J.ht)[2 * (int64_t)s] = 0;
        }
    }
}

} // namespace

// Which programs run this way: selections over at most DIM_COLS columns from
// flags that start all true, then one build; at most one flag buffer stored,
// no column stored.  A build side of DIM_MAX_ROWS rows or more fills the chip
// by itself and keeps its own compiled and tuned kernel.
bool dim_job(const FProgram &p, int64_t n, DimJob &J)
{
    if (n <= 0 || n >= DIM_MAX_ROWS || p.ninstr < 1 || p.ninstr > DIM_INSTRS + 1 || p.sum_acc || p.gb.k) return false;
    J = DimJob{};
    auto column = [&](int8_t reg, const int32_t *mem, uint8_t &out) {
        if (reg >= F_PF_BASE) mem = p.pf_mem[reg - F_PF_BASE];
        else if (reg >= 0) return false; // a value the program makes
        if (!mem) return false;
        for (int c = 0; c < J.ncols; c++)
            if (J.col[c] == mem) {
                out = (uint8_t)c;
                return true;
            }
        if (J.ncols == DIM_COLS) return false;
        out = (uint8_t)J.ncols;
        J.col[J.ncols++] = mem;
        return true;
    };
    for (int f = 0; f < F_MAX_FLAGS; f++) {
        if (p.flag_init[f] == FF_LOAD) return false;
        if (p.flag_init[f] == FF_TRUE) J.init |= 15u << (4 * f);
        if (!p.flag_store[f]) continue;
        if (J.store) return false;
        J.store = p.flag_store[f];
        J.store_reg = (uint8_t)f;
    }
    for (int i = 0; i + 1 < p.ninstr; i++) {
        const FInstr &I = p.ins[i];
        DimInstr &D = J.ins[J.ninstr++];
        D = {I.kind, I.cmp, I.logic, I.fin, I.fout, I.floc, 0, 0, I.lit, I.lit2};
        switch (I.kind) {
        case FK_LOGICAL: break;
        case FK_SEL_LIT:
        case FK_SEL_RANGE:
        case FK_SEL_IN2:
            if (!column(I.va, I.a, D.a)) return false;
            break;
        case FK_SEL_COL:
            if (!column(I.va, I.a, D.a) || !column(I.vb, I.b, D.b)) return false;
            break;
        default: return false;
        }
    }
    const FInstr &B = p.ins[p.ninstr - 1];
    if (B.kind != FK_BUILD_KEYS && B.kind != FK_BUILD_KEYVALS) return false;
    J.pairs = B.kind == FK_BUILD_KEYVALS;
    if (!column(B.va, B.a, J.key)) return false;
    if (J.pairs && !column(B.vb, B.b, J.val)) return false;
    J.fin = B.fin;
    J.ht = const_cast<void *>(B.ht);
    J.ht_min = B.ht_min;
    J.ht_len = B.ht_len;
    J.n = (int32_t)n;
    J.vec = (uint8_t)(p.vec != 0);
    return true;
}

template <int N> static void launch_jobs(const DimJob *jobs, int n, hipStream_t s)
{
    DimJobs<N> J{};
    std::fill(std::begin(J.first), std::end(J.first), UINT32_MAX);
    uint32_t blocks = 0;
    for (int i = 0; i < n; i++) {
        J.first[i] = blocks;
        J.job[i] = jobs[i];
        J.nblocks[i] = (uint32_t)std::min<int64_t>((jobs[i].n + DIM_STEP - 1) / DIM_STEP, DIM_MAX_BLOCKS);
        blocks += J.nblocks[i];
    }
    hipLaunchKernelGGL((k_dim_builds<N>), dim3(blocks), dim3(DIM_BLOCK), 0, s, J);
    hip_check(hipGetLastError(), "dim_builds");
}

int launch_dim_builds(const DimJob *jobs, size_t njobs, hipStream_t s)
{
    int launches = 0;
    for (size_t at = 0; at < njobs; at += DIM_JOBS, launches++) {
        const int n = (int)std::min<size_t>(DIM_JOBS, njobs - at);
        if (n <= DIM_JOBS_SMALL) launch_jobs<DIM_JOBS_SMALL>(jobs + at, n, s);
        else launch_jobs<DIM_JOBS>(jobs + at, n, s);
    }
    return launches;
}

} // namespace sdb
