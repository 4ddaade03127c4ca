// Plan analysis and the plan walk: operations/preprocessing.cpp:14-275 and
// executor/ddor_executor.cpp:22-245.
#include <cstring>
#include <deque>
#include <iostream>
#include <set>

#include "engine.hpp"

namespace sdb {

// kernels/types.cpp:3-21
const std::map<std::string, int> TABLE_COLUMN_NUMBERS = {
    {"lineorder", 17}, {"part", 9}, {"supplier", 7}, {"customer", 8}, {"ddate", 17}};
const std::map<std::string, std::vector<int>> TABLE_COLUMN_INDICES = {
    {"lineorder", {2, 3, 4, 5, 8, 9, 11, 12, 13}},
    {"part", {0, 2, 3, 4}},
    {"supplier", {0, 3, 4, 5}},
    {"customer", {0, 3, 4, 5}},
    {"ddate", {0, 4, 5}}};

namespace {

int column_count(const std::string &table)
{
    auto it = TABLE_COLUMN_NUMBERS.find(table);
    if (it == TABLE_COLUMN_NUMBERS.end()) throw std::invalid_argument("unknown table " + table);
    return it->second;
}

void expression_columns(const ExprType &e, std::set<int64_t> &out)
{
    if (e.exprType == ExprOption::COLUMN) out.insert(e.input);
    else if (e.exprType == ExprOption::EXPR)
        for (const ExprType &o : e.operands) expression_columns(o, out);
}

} // namespace

std::vector<int> dag_topological_sort(const PlanResult &plan)
{
    const size_t n = plan.rels.size();
    std::vector<std::vector<char>> dag(n, std::vector<char>(n, 0));
    std::deque<int> S;
    auto edge = [&](int64_t a, int64_t b) {
        if (a < 0 || b < 0 || a >= (int64_t)n || b >= (int64_t)n) throw std::invalid_argument("plan: bad rel input");
        dag[a][b] = 1;
    };
    for (const RelNode &rel : plan.rels) {
        switch (rel.relOp) {
        case RelNodeType::TABLE_SCAN: S.push_front((int)rel.id); break;
        case RelNodeType::FILTER:
        case RelNodeType::PROJECT:
        case RelNodeType::AGGREGATE:
        case RelNodeType::SORT: edge(rel.id - 1, rel.id); break;
        case RelNodeType::JOIN:
            if (rel.inputs.size() != 2) return {};
            edge(rel.inputs[0], rel.id);
            edge(rel.inputs[1], rel.id);
            break;
        default: return {};
        }
    }
    std::vector<int> sorted;
    while (!S.empty()) {
        const int node = S.back();
        S.pop_back();
        const RelNode &r = plan.rels[node];
        // the lineorder scan waits until it is the only source left (60-66)
        if (!S.empty() && r.relOp == RelNodeType::TABLE_SCAN && r.tables.size() > 1 && r.tables[1] == "lineorder") {
            S.push_front(node);
            continue;
        }
        sorted.push_back(node);
        for (size_t i = 0; i < n; i++) {
            if (!dag[node][i]) continue;
            dag[node][i] = 0;
            bool inbound = false;
            for (size_t j = 0; j < n && !inbound; j++) inbound = dag[j][i] != 0;
            if (!inbound) S.push_front((int)i);
        }
    }
    if (sorted.size() != n) return {};
    return sorted;
}

ExecutionInfo parse_execution_info(const PlanResult &plan)
{
    ExecutionInfo info;
    using Info = std::vector<std::pair<std::string, int>>;
    std::vector<Info> ops;
    auto at = [](const Info &v, int64_t i) -> const std::pair<std::string, int> & {
        if (i < 0 || i >= (int64_t)v.size()) throw std::invalid_argument("plan: column reference out of range");
        return v[i];
    };
    for (const RelNode &rel : plan.rels) {
        switch (rel.relOp) {
        case RelNodeType::TABLE_SCAN: {
            if (rel.tables.size() < 2) throw std::invalid_argument("plan: TABLE_SCAN needs [schema, table]");
            Info t;
            for (int i = 0; i < column_count(rel.tables[1]); i++) t.emplace_back(rel.tables[1], i);
            info.loaded_columns[rel.tables[1]];
            ops.push_back(t);
            break;
        }
        case RelNodeType::FILTER: {
            if (ops.empty()) throw std::invalid_argument("plan: FILTER without input");
            Info t = ops.back();
            std::set<int64_t> cols;
            expression_columns(rel.condition, cols);
            for (int64_t c : cols) info.loaded_columns[at(t, c).first].push_back(at(t, c).second);
            ops.push_back(t);
            break;
        }
        case RelNodeType::PROJECT: {
            if (ops.empty()) throw std::invalid_argument("plan: PROJECT without input");
            const Info last = ops.back();
            Info t;
            for (const ExprType &e : rel.exprs) {
                std::set<int64_t> cols;
                expression_columns(e, cols);
                for (int64_t c : cols) info.loaded_columns[at(last, c).first].push_back(at(last, c).second);
                if (!cols.empty()) t.push_back(at(last, *cols.begin()));
            }
            ops.push_back(t);
            break;
        }
        case RelNodeType::AGGREGATE: {
            if (ops.empty()) throw std::invalid_argument("plan: AGGREGATE without input");
            const Info last = ops.back();
            Info t;
            for (int64_t g : rel.group) {
                const auto &tc = at(last, g);
                info.loaded_columns[tc.first].push_back(tc.second);
                t.push_back(tc);
                info.group_by_columns[tc.first] = tc.second;
            }
            for (const AggType &a : rel.aggs) {
                for (int64_t c : a.operands) info.loaded_columns[at(last, c).first].push_back(at(last, c).second);
                if (!a.operands.empty()) t.push_back(at(last, a.operands[0]));
            }
            ops.push_back(t);
            break;
        }
        case RelNodeType::JOIN: {
            if (rel.inputs.size() != 2) throw std::invalid_argument("plan: JOIN needs two inputs");
            for (int64_t in : rel.inputs)
                if (in < 0 || in >= (int64_t)ops.size()) throw std::invalid_argument("plan: JOIN input out of range");
            Info t = ops[rel.inputs[0]];
            const Info &r = ops[rel.inputs[1]];
            t.insert(t.end(), r.begin(), r.end());
            ops.push_back(t);
            break;
        }
        case RelNodeType::SORT: {
            if (ops.empty()) throw std::invalid_argument("plan: SORT without input");
            ops.push_back(ops.back());
            break;
        }
        default: std::cerr << "Unsupported RelNodeType" << std::endl; break;
        }
    }
    info.dag_order = dag_topological_sort(plan);
    return info;
}

FinalTable run_ddor_plan(Engine &eng, const PlanResult &plan)
{
    const ExecutionInfo info = parse_execution_info(plan);
    if (info.dag_order.empty()) throw std::runtime_error("DAG topological sort failed");
    std::vector<int> output_table(plan.rels.size(), -1);
    std::deque<TransientTable> tts;
    for (const RelNode &rel : plan.rels) {
        if (rel.relOp != RelNodeType::TABLE_SCAN) continue;
        Table *t = eng.find_table(rel.tables[1]);
        if (!t) throw std::invalid_argument("Table " + rel.tables[1] + " not found among loaded tables.");
        TransientTable &tt = tts.emplace_back(eng, t);
        auto gb = info.group_by_columns.find(rel.tables[1]);
        if (gb != info.group_by_columns.end()) tt.set_group_by_column(gb->second);
        output_table[rel.id] = (int)tts.size() - 1;
    }
    auto input_of = [&](int64_t id) -> TransientTable & {
        if (id < 0 || id >= (int64_t)output_table.size() || output_table[id] < 0)
            throw std::invalid_argument("plan: operator input has no table");
        return tts[output_table[id]];
    };
    for (int id : info.dag_order) {
        const RelNode &rel = plan.rels[id];
        switch (rel.relOp) {
        case RelNodeType::TABLE_SCAN: break;
        case RelNodeType::FILTER:
            input_of(id - 1).apply_filter(rel.condition, "");
            output_table[id] = output_table[id - 1];
            break;
        case RelNodeType::PROJECT:
            input_of(id - 1).apply_project(rel.exprs);
            output_table[id] = output_table[id - 1];
            break;
        case RelNodeType::AGGREGATE:
            if (rel.aggs.empty()) throw std::invalid_argument("plan: AGGREGATE without aggs");
            input_of(id - 1).apply_aggregate(rel.aggs[0], rel.group);
            output_table[id] = output_table[id - 1];
            break;
        case RelNodeType::JOIN:
            input_of(rel.inputs[0]).apply_join(input_of(rel.inputs[1]), rel);
            output_table[id] = output_table[rel.inputs[0]];
            break;
        case RelNodeType::SORT: output_table[id] = output_table[id - 1]; break;
        default: std::cerr << "RelNodeType not yet supported in DDOR." << std::endl; break;
        }
    }
    TransientTable &final_table = input_of((int64_t)plan.rels.size() - 1);
    final_table.execute_pending_kernels(false);
    if (!eng.capture.active) eng.flush_builds();

    FinalTable t;
    t.nrows = final_table.get_nrows();
    final_table.selection(t.flags, t.seen);
    for (Column *c : final_table.get_columns()) {
        if (!c || !c->loaded || !c->data) continue;
        t.cols.push_back({c->data, c->is_aggregate, std::min(t.nrows, c->nrows)});
    }
    return t;
}

void Engine::print_marks()
{
    if (marks.empty()) return;
    const auto t0 = marks.front().first;
    std::string line = "[step]";
    for (const auto &m : marks) {
        char buf[64];
        snprintf(buf, sizeof(buf), " %.1f", std::chrono::duration<double, std::micro>(m.first - t0).count());
        line += buf;
        line += " " + m.second + ";";
    }
    fprintf(stderr, "%s\n", line.c_str());
    marks.clear();
}

void Engine::wait_stream()
{
    if (!sync_ev) SDB_HIP(hipEventCreateWithFlags(&sync_ev, hipEventDisableTiming));
    hipEvent_t ev = stop_at_wait ? ev_stop : sync_ev;
    SDB_HIP(hipEventRecord(ev, stream));
    hipError_t e;
    while ((e = hipEventQuery(ev)) == hipErrorNotReady) {
    }
    SDB_HIP(e);
    if (stop_at_wait) stop_recorded = true;
}

// A result's largest possible size may ask for tens of megabytes that the next
// thousands of results do without: a buffer four times larger than any of the
// last PINNED_WINDOW requests goes back.  The call that gives 50 MB back takes
// 0.4 to 0.9 ms, the next one that needs them 0.3 to 0.5; over 4,096 calls of 65 us
// that is at most 0.5 % (over 256 it was up to 8).
void *Engine::pinned_buffer(size_t bytes)
{
    constexpr size_t PINNED_MIN = 1 << 20;
    constexpr int PINNED_WINDOW = 4096;
    pinned_most = std::max(pinned_most, bytes);
    bool wasteful = false;
    if (++pinned_calls >= PINNED_WINDOW) {
        wasteful = pinned_bytes > 4 * std::max(pinned_most, PINNED_MIN);
        bytes = wasteful ? pinned_most : bytes;
        pinned_calls = 0;
        pinned_most = 0;
    }
    if (bytes > pinned_bytes || wasteful) {
        if (pinned) SDB_HIP(hipHostFree(pinned));
        pinned = nullptr;
        pinned_bytes = 0;
        const size_t want = std::max(bytes, PINNED_MIN);
        SDB_HIP(hipHostMalloc(&pinned, want, hipHostMallocDefault));
        pinned_bytes = want;
    }
    return pinned;
}

namespace {

// Group-by results of at least this many slots come back compacted on the
// device: only their selected rows cross PCIe and reach host memory.
constexpr uint64_t RESULT_SPARSE_MIN_ROWS = 1u << 15;

bool sparse_result(const FinalTable &t)
{
    if (t.nrows < RESULT_SPARSE_MIN_ROWS || t.nrows >= (1ull << 31) || (!t.flags && !t.seen) ||
        t.cols.size() > (size_t)GATHER_MAX_COLS)
        return false;
    for (const FinalTable::Col &c : t.cols)
        if (c.is_u64) return true;
    return false;
}

// Device-to-host copies through the engine's pinned staging buffer: every
// copy queued, one wait for the stream, then into host memory.  Up to
// PACK_DIRECT_BYTES in all, one kernel writes the arrays straight into the
// staging buffer; up to PACK_MAX_BYTES they are packed on the device first and
// cross PCIe in one transfer.  (A q2.x result, 119 KB in four arrays: packing,
// transfer and the gap between them 8 us, the direct writes 4.)
constexpr size_t PACK_DIRECT_BYTES = size_t(1) << 20;
constexpr size_t PACK_MAX_BYTES = size_t(64) << 20;
struct HostCopies {
    struct Part {
        const void *src;
        void *dst;
        size_t off, bytes;
        PackKind kind;
    };
    std::vector<Part> parts;
    size_t total = 0;
    void add(const void *src, void *dst, size_t bytes, PackKind kind = PACK_COPY)
    {
        if (!bytes) return;
        total = (total + 15) / 16 * 16;
        parts.push_back({src, dst, total, bytes, kind});
        total += bytes;
    }
    void pack(Engine &eng, uint8_t *to)
    {
        PackParts pk{};
        for (size_t i = 0; i < parts.size(); i++) {
            pk.src[pk.n] = static_cast<const uint8_t *>(parts[i].src);
            pk.off[pk.n] = parts[i].off;
            pk.bytes[pk.n] = parts[i].bytes;
            pk.kind[pk.n] = parts[i].kind;
            if (++pk.n == PACK_MAX_PARTS || i + 1 == parts.size()) {
                launch_pack_parts(pk, to, eng.stream);
                eng.launches++;
                pk.n = 0;
            }
        }
    }
    // queues the copies into `host` (total bytes of pinned memory)
    void queue(Engine &eng, uint8_t *host)
    {
        if (total <= PACK_DIRECT_BYTES) {
            pack(eng, host);
            return;
        }
        if (total <= PACK_MAX_BYTES) {
            uint8_t *dev = eng.mm->alloc<uint8_t>(total);
            pack(eng, dev);
            SDB_HIP(hipMemcpyAsync(host, dev, total, hipMemcpyDeviceToHost, eng.stream));
            return;
        }
        for (const Part &p : parts) {
            if (p.kind == PACK_TRUE) {
                std::memset(host + p.off, 1, p.bytes);
                continue;
            }
            const void *src = p.src;
            if (p.kind == PACK_SEEN) {
                uint8_t *flags = eng.mm->alloc<uint8_t>(p.bytes);
                launch_seen_to_flags(static_cast<const uint32_t *>(p.src), flags, p.bytes, eng.stream);
                eng.launches++;
                src = flags;
            }
            SDB_HIP(hipMemcpyAsync(host + p.off, src, p.bytes, hipMemcpyDeviceToHost, eng.stream));
        }
    }
    void wait(Engine &eng)
    {
        eng.mark("result wait");
        eng.wait_stream();
        eng.mark("result ready");
    }
    // after the wait
    void deliver(const uint8_t *host)
    {
        for (const Part &p : parts) std::memcpy(p.dst, host + p.off, p.bytes);
        parts.clear();
        total = 0;
    }
};

// Sparse tables whose largest possible result fits the staging buffer
// (SPARSE_STAGE_MAX for all of a call's) have their selected rows written
// there by the kernels that find them.
constexpr size_t SPARSE_STAGE_MAX = size_t(64) << 20;

size_t sparse_stage_bytes(const FinalTable &t)
{
    size_t b = 16 + (t.nrows * 4 + 15) / 16 * 16; // count, row ids
    for (const FinalTable::Col &c : t.cols) b += (t.nrows * (c.is_u64 ? 8 : 4) + 15) / 16 * 16;
    return b;
}

} // namespace

std::vector<ResultTable> copy_results(Engine &eng, const std::vector<FinalTable> &ts)
{
    // host copies of the final tables (the materialize_host_view +
    // save_result path, executor/result_writer.cpp:28-67), all tables in one
    // wait for the stream (two when a large group-by does not fit the staging)
    std::vector<ResultTable> out(ts.size());
    HostCopies copies;
    std::vector<size_t> sparse, staged; // staged: written into the staging buffer by the device
    size_t stage_total = 0;
    for (size_t i = 0; i < ts.size(); i++) {
        const FinalTable &t = ts[i];
        if (!sparse_result(t)) continue;
        out[i].sparse = true;
        const size_t b = sparse_stage_bytes(t);
        if (t.nrows <= SPARSE_MAX_ROWS && stage_total + b <= SPARSE_STAGE_MAX) {
            staged.push_back(i);
            stage_total += b;
        } else {
            sparse.push_back(i);
        }
    }
    // the other large group-by tables: the selected row ids, compacted in row
    // order on the device; their counts come back with the dense tables
    std::vector<int32_t *> ids(ts.size(), nullptr);
    std::vector<uint32_t> counts(sparse.size(), 0);
    if (!sparse.empty()) {
        uint32_t *d_counts = eng.mm->alloc<uint32_t>(sparse.size());
        for (size_t j = 0; j < sparse.size(); j++) {
            const FinalTable &t = ts[sparse[j]];
            const uint8_t *flags = t.flags;
            if (!flags) {
                eng.registry.check(t.seen, t.nrows * 4, "result group-by slots");
                uint8_t *f = eng.mm->alloc<uint8_t>(t.nrows);
                launch_seen_to_flags(t.seen, f, t.nrows, eng.stream);
                eng.launches++;
                flags = f;
            }
            eng.registry.check(flags, t.nrows, "result flags");
            int32_t *row_ids = eng.mm->alloc<int32_t>(t.nrows);
            uint32_t *tiles = eng.mm->alloc<uint32_t>((uint64_t)std::max<int64_t>(compact_tiles((int64_t)t.nrows), 1));
            launch_compact_into(flags, (int64_t)t.nrows, row_ids, d_counts + j, tiles, eng.stream);
            eng.launches += 3;
            ids[sparse[j]] = row_ids;
        }
        copies.add(d_counts, counts.data(), counts.size() * 4);
    }
    for (size_t i = 0; i < ts.size(); i++) {
        const FinalTable &t = ts[i];
        ResultTable &res = out[i];
        res.nrows = t.nrows;
        for (const FinalTable::Col &c : t.cols) {
            ResultTable::Col rc;
            rc.is_u64 = c.is_u64;
            res.cols.push_back(std::move(rc));
        }
        if (res.sparse) continue;
        res.flags.resize(res.nrows);
        if (res.nrows) {
            if (t.flags) eng.registry.check(t.flags, res.nrows, "result flags");
            else if (t.seen) eng.registry.check(t.seen, res.nrows * 4, "result group-by slots");
            copies.add(t.flags ? (const void *)t.flags : (const void *)t.seen, res.flags.data(), res.nrows,
                       t.flags ? PACK_COPY : t.seen ? PACK_SEEN : PACK_TRUE);
        }
        for (size_t c = 0; c < t.cols.size(); c++) {
            const FinalTable::Col &fc = t.cols[c];
            ResultTable::Col &rc = res.cols[c];
            const uint64_t elem = rc.is_u64 ? 8 : 4;
            if (rc.is_u64) rc.u64.assign(res.nrows, 0);
            else rc.i32.assign(res.nrows, 0);
            if (fc.rows) {
                eng.registry.check(fc.data, fc.rows * elem, "result column");
                copies.add(fc.data, rc.is_u64 ? (void *)rc.u64.data() : (void *)rc.i32.data(), fc.rows * elem);
            }
        }
    }
    // one staging buffer: the packed arrays, then the staged sparse tables
    const size_t stage_off = (copies.total + 15) / 16 * 16;
    uint8_t *host = static_cast<uint8_t *>(eng.pinned_buffer(std::max<size_t>(stage_off + stage_total, 1)));
    std::vector<SparseTable> st(staged.size());
    uint8_t *at = host + stage_off;
    auto take = [&at](size_t bytes) {
        uint8_t *p = at;
        at += (bytes + 15) / 16 * 16;
        return p;
    };
    for (size_t j = 0; j < staged.size(); j++) {
        const FinalTable &t = ts[staged[j]];
        SparseTable &s = st[j];
        s = SparseTable{};
        if (t.flags) eng.registry.check(t.flags, t.nrows, "result flags");
        else eng.registry.check(t.seen, t.nrows * 4, "result group-by slots");
        s.flags = t.flags;
        s.seen = t.seen;
        s.rows = (uint32_t)t.nrows;
        s.counts = eng.mm->alloc<uint32_t>(sparse_tiles(t.nrows));
        s.count = reinterpret_cast<uint32_t *>(take(4));
        s.ids = reinterpret_cast<uint32_t *>(take(t.nrows * 4));
        s.ncols = (int32_t)t.cols.size();
        for (size_t c = 0; c < t.cols.size(); c++) {
            const FinalTable::Col &fc = t.cols[c];
            const uint64_t elem = fc.is_u64 ? 8 : 4;
            if (fc.rows) eng.registry.check(fc.data, fc.rows * elem, "result column");
            s.src[c] = fc.data;
            s.src_rows[c] = (uint32_t)std::min<uint64_t>(fc.rows, t.nrows);
            if (fc.is_u64) s.is_u64 |= 1u << c;
            s.dst[c] = take(t.nrows * elem);
        }
    }
    if (!copies.parts.empty()) copies.queue(eng, host);
    if (!st.empty()) eng.launches += launch_sparse_tables(st.data(), st.size(), eng.stream);
    copies.wait(eng);
    copies.deliver(host);
    for (ResultTable &res : out)
        if (!res.sparse && res.nrows < RESULT_SPARSE_MIN_ROWS) res.list_selected();
    for (size_t j = 0; j < staged.size(); j++) {
        ResultTable &res = out[staged[j]];
        const SparseTable &s = st[j];
        const uint32_t k = *s.count;
        if (k > s.rows) fail(SDB_ERR_RUNTIME, "result compaction: selected count out of range");
        res.sel.assign(s.ids, s.ids + k);
        for (size_t c = 0; c < res.cols.size(); c++) {
            ResultTable::Col &rc = res.cols[c];
            if (rc.is_u64) rc.u64.assign(static_cast<const uint64_t *>(s.dst[c]), static_cast<const uint64_t *>(s.dst[c]) + k);
            else rc.i32.assign(static_cast<const int32_t *>(s.dst[c]), static_cast<const int32_t *>(s.dst[c]) + k);
        }
    }
    // the large ones that were not staged: every column gathered at the
    // selected rows on the device, then copied
    for (size_t j = 0; j < sparse.size(); j++) {
        const FinalTable &t = ts[sparse[j]];
        ResultTable &res = out[sparse[j]];
        const uint32_t k = counts[j];
        if (k > t.nrows) fail(SDB_ERR_RUNTIME, "result compaction: selected count out of range");
        res.sel.resize(k);
        if (!k) continue;
        GatherCols g{};
        g.ncols = (int32_t)t.cols.size();
        for (size_t c = 0; c < t.cols.size(); c++) {
            const FinalTable::Col &fc = t.cols[c];
            ResultTable::Col &rc = res.cols[c];
            const uint64_t elem = fc.is_u64 ? 8 : 4;
            if (fc.rows) eng.registry.check(fc.data, fc.rows * elem, "result column");
            g.src[c] = fc.data;
            g.src_rows[c] = fc.rows;
            if (fc.is_u64) g.is_u64 |= 1u << c;
            void *d = eng.mm->alloc<uint8_t>((uint64_t)k * elem);
            g.dst[c] = d;
            if (fc.is_u64) rc.u64.resize(k);
            else rc.i32.resize(k);
            copies.add(d, fc.is_u64 ? (void *)rc.u64.data() : (void *)rc.i32.data(), (size_t)k * elem);
        }
        launch_gather_cols(g, ids[sparse[j]], (int64_t)k, eng.stream);
        eng.launches++;
        copies.add(ids[sparse[j]], res.sel.data(), (size_t)k * 4);
    }
    if (!copies.parts.empty()) {
        host = static_cast<uint8_t *>(eng.pinned_buffer(copies.total));
        copies.queue(eng, host);
        copies.wait(eng);
        copies.deliver(host);
    }
    return out;
}

ResultTable copy_result(Engine &eng, const FinalTable &t) { return std::move(copy_results(eng, {t})[0]); }

void ResultTable::list_selected()
{
    uint64_t r = 0;
    for (; r + 8 <= flags.size(); r += 8) { // mostly empty group-by slots: eight at a time
        uint64_t w;
        std::memcpy(&w, flags.data() + r, 8);
        if (!w) continue;
        for (uint64_t k = r; k < r + 8; k++)
            if (flags[k]) sel.push_back((uint32_t)k);
    }
    for (; r < flags.size(); r++)
        if (flags[r]) sel.push_back((uint32_t)r);
    listed = true;
}

void ResultTable::selected_to(uint8_t *host) const
{
    const uint64_t k = selected();
    selected_rows_to(reinterpret_cast<uint64_t *>(host));
    host += 8 * k;
    for (size_t c = 0; c < cols.size(); c++) {
        col_selected_to((int)c, host);
        host += ((cols[c].is_u64 ? 8 : 4) * k + 7) / 8 * 8;
    }
}

uint64_t ResultTable::selected() const
{
    if (sparse || listed) return sel.size();
    uint64_t n = 0;
    for (uint8_t f : flags) n += f != 0;
    return n;
}

void ResultTable::flags_to(uint8_t *host) const
{
    if (!sparse) {
        std::memcpy(host, flags.data(), flags.size());
        return;
    }
    std::memset(host, 0, nrows);
    for (uint32_t r : sel) host[r] = 1;
}

void ResultTable::col_to(int c, void *host) const
{
    const Col &col = cols[c];
    if (!sparse) {
        if (col.is_u64) std::memcpy(host, col.u64.data(), col.u64.size() * 8);
        else std::memcpy(host, col.i32.data(), col.i32.size() * 4);
        return;
    }
    if (col.is_u64) {
        uint64_t *h = static_cast<uint64_t *>(host);
        std::memset(h, 0, nrows * 8);
        for (size_t j = 0; j < sel.size(); j++) h[sel[j]] = col.u64[j];
    } else {
        int32_t *h = static_cast<int32_t *>(host);
        std::memset(h, 0, nrows * 4);
        for (size_t j = 0; j < sel.size(); j++) h[sel[j]] = col.i32[j];
    }
}

void ResultTable::selected_rows_to(uint64_t *host) const
{
    if (sparse || listed) {
        for (size_t j = 0; j < sel.size(); j++) host[j] = sel[j];
        return;
    }
    uint64_t j = 0;
    for (uint64_t r = 0; r < flags.size(); r++)
        if (flags[r]) host[j++] = r;
}

void ResultTable::col_selected_to(int c, void *host) const
{
    const Col &col = cols[c];
    if (sparse) {
        if (col.is_u64) std::memcpy(host, col.u64.data(), col.u64.size() * 8);
        else std::memcpy(host, col.i32.data(), col.i32.size() * 4);
        return;
    }
    if (listed) {
        if (col.is_u64)
            for (size_t j = 0; j < sel.size(); j++) static_cast<uint64_t *>(host)[j] = col.u64[sel[j]];
        else
            for (size_t j = 0; j < sel.size(); j++) static_cast<int32_t *>(host)[j] = col.i32[sel[j]];
        return;
    }
    uint64_t j = 0;
    for (uint64_t r = 0; r < flags.size(); r++) {
        if (!flags[r]) continue;
        if (col.is_u64) static_cast<uint64_t *>(host)[j++] = col.u64[r];
        else static_cast<int32_t *>(host)[j++] = col.i32[r];
    }
}

ResultTable execute_ddor_plan(Engine &eng, const PlanResult &plan) { return copy_result(eng, run_ddor_plan(eng, plan)); }

} // namespace sdb
