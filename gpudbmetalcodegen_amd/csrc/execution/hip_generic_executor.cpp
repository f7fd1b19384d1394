#include "hip_generic_executor.h"

#include "gdb/gdb_kernels.h"

#include <cctype>

#include <algorithm>
#include <chrono>
#include <cstring>

namespace gdb {
namespace codegen {

namespace {

void check(gdb_status st, const std::string& what) {
    if (st != GDB_OK) throw std::runtime_error(what + ": " + gdb_last_error());
}

}  // namespace

HipGenericExecutor::HipGenericExecutor(gdb_ctx ctx, gdb_stream stream)
    : ctx_(ctx), stream_(stream ? stream : gdb_default_stream(ctx)) {
    gdb_device_info_t info;
    check(gdb_device_info(ctx_, &info), "gdb_device_info");
    cuCount_ = info.cu_count;
}

HipGenericExecutor::~HipGenericExecutor() {
    releaseAllocatedBuffers();
    for (auto e : events_) gdb_event_destroy(e);
    dropPinned();
}

uint64_t* HipGenericExecutor::ensurePinned(size_t bytes) {
    if (bytes > pinnedBytes_) {
        check(gdb_stream_sync(stream_), "gdb_stream_sync");  // no copy into the old block is in flight
        pinnedInFlight_ = false;
        dropPinned();
        void* h = nullptr;
        if (bytes <= GDB_PINNED_BLOCK)
            check(gdb_host_take_block(&h), "gdb_host_take_block");
        else
            check(gdb_host_alloc_pinned(bytes, &h), "gdb_host_alloc_pinned");
        pinned_ = static_cast<uint64_t*>(h);
        pinnedBytes_ = std::max<size_t>(bytes, GDB_PINNED_BLOCK);
    }
    pinnedInFlight_ = true;  // until the caller has waited for what it enqueues
    return pinned_;
}

void HipGenericExecutor::dropPinned() {
    // a block something may still write (a failed run) is freed, which waits, and not shared again
    if (pinnedBytes_ == GDB_PINNED_BLOCK && !pinnedInFlight_)
        gdb_host_give_block(pinned_);
    else if (pinned_)
        gdb_host_free_pinned(pinned_);
    pinned_ = nullptr;
    pinnedBytes_ = 0;
}

void HipGenericExecutor::syncStream() {
    check(gdb_stream_sync(stream_), "gdb_stream_sync");
    pinnedInFlight_ = false;
}

void HipGenericExecutor::registerTable(const std::string& table, uint64_t rows) {
    TableInfo& t = tables_[table];
    t.rows = rows;
    sizes_.registerSymbol(tableSizeName(table), rows);
    if (t.registered && rows <= t.mostRows) return;
    t.registered = true;
    t.mostRows = rows;
    sizes_.registerSymbol(tableMaxSizeName(table), rows);
}

void HipGenericExecutor::registerTableColumn(const std::string& table, const std::string& column, const void* devptr) {
    if (reinterpret_cast<uintptr_t>(devptr) % 16 != 0)
        throw std::runtime_error("registerTableColumn: column " + column + " must be 16-byte aligned");
    tables_[table].columns[column] = devptr;
}

void HipGenericExecutor::registerBuffer(const std::string& name, void* devptr, size_t bytes) {
    auto it = buffers_.find(name);
    if (it != buffers_.end() && it->second.owned) gdb_free(ctx_, it->second.ptr);
    buffers_[name] = Buffer{devptr, bytes, false};
}

void HipGenericExecutor::registerBufferTable(const std::string& table, const std::string& column,
                                             const std::string& buffer, const std::string& rowsExpr) {
    for (auto& bt : bufferTables_)
        if (bt.table == table && bt.column == column) {
            bt.buffer = buffer;
            bt.rowsExpr = rowsExpr;
            return;
        }
    bufferTables_.push_back({table, column, buffer, rowsExpr});
}

void HipGenericExecutor::registerSymbol(const std::string& name, uint64_t value) { sizes_.registerSymbol(name, value); }

bool HipGenericExecutor::tryGetSymbol(const std::string& name, uint64_t& out) const {
    if (!sizes_.hasSymbol(name)) return false;
    out = sizes_.getSymbol(name);
    return true;
}

void HipGenericExecutor::registerScalarInt(const std::string& name, int64_t value) { scalars_[name] = value; }

void HipGenericExecutor::setPhaseHook(const std::string& phase, std::function<void(HipGenericExecutor&)> hook,
                                      const std::string& readBuffer, size_t readOffset, size_t readBytes) {
    if (readBytes > 4096) throw std::runtime_error("setPhaseHook: read-ahead of at most 4096 bytes");
    hooks_[phase] = Hook{std::move(hook), readBuffer, readOffset, readBytes};
}

HipGenericExecutor::Buffer& HipGenericExecutor::ensureBuffer(const HipParamBinding& b) {
    auto it = buffers_.find(b.name);
    if (b.sizeExpr.empty()) {
        if (it == buffers_.end())
            throw std::runtime_error("executor: buffer '" + b.name + "' is neither registered nor sized by the plan");
        return it->second;
    }
    const uint64_t elems = sizes_.resolve(b.sizeExpr);
    const size_t bytes = std::max<size_t>(static_cast<size_t>(elems) * b.elemBytes, 16);
    if (it != buffers_.end()) {
        if (!it->second.owned || it->second.bytes >= bytes) return it->second;
        check(gdb_free(ctx_, it->second.ptr), "gdb_free");
        buffers_.erase(it);
    }
    Buffer nb;
    nb.bytes = ((bytes + 255) / 256) * 256;
    check(gdb_alloc(ctx_, nb.bytes, &nb.ptr), "gdb_alloc(" + b.name + ", " + std::to_string(nb.bytes) + " bytes)");
    nb.owned = true;
    return buffers_[b.name] = nb;
}

void HipGenericExecutor::resolveBufferTables() {
    for (const auto& bt : bufferTables_) {
        auto it = buffers_.find(bt.buffer);
        if (it == buffers_.end()) continue;
        tables_[bt.table].columns[bt.column] = it->second.ptr;
        const uint64_t rows = sizes_.resolve(bt.rowsExpr);
        tables_[bt.table].rows = rows;
        sizes_.registerSymbol(tableSizeName(bt.table), rows);
    }
}

std::unordered_map<std::string, const HipParamBinding*> HipGenericExecutor::initSpecs(const HipCodegen& cg) const {
    std::unordered_map<std::string, const HipParamBinding*> spec;
    for (const auto& p : cg.getPhases())
        for (const auto& b : p.bindings)
            if (b.kind == HipParamKind::DeviceBuffer && b.init != InitKind::None && !spec.count(b.name))
                spec[b.name] = &b;
    return spec;
}

namespace {

// A size and pattern the multi-buffer fill takes (gdb_fill_multi_async):
// whole 8-byte words, a pattern of 1, 2 or 4 bytes or 1..4 words dividing it.
bool multiFillable(size_t bytes, int pl) {
    if (bytes % 8 != 0 || pl < 1) return false;
    if (pl == 1 || pl == 2 || pl == 4) return true;
    return pl % 8 == 0 && pl <= 32 && bytes % static_cast<size_t>(pl) == 0;
}

// The shortest prefix of a fill pattern that repeats to the whole pattern,
// among the lengths the multi-buffer fill takes (1, 2, 4 bytes, 1..4 words):
// a 16-word all-zero bucket pattern fills as one zero word. The pattern
// itself when none does.
std::vector<uint8_t> shortestPeriod(const std::vector<uint8_t>& pat) {
    for (size_t p : {1, 2, 4, 8, 16, 24, 32}) {
        if (p >= pat.size()) break;
        if (pat.size() % p != 0) continue;
        bool periodic = true;
        for (size_t i = p; i < pat.size() && periodic; ++i) periodic = pat[i] == pat[i % p];
        if (periodic) return std::vector<uint8_t>(pat.begin(), pat.begin() + static_cast<long>(p));
    }
    return pat;
}

bool mentionsSymbol(const std::string& expr, const std::string& sym) {
    size_t pos = 0;
    while ((pos = expr.find(sym, pos)) != std::string::npos) {
        const bool startOk = pos == 0 || !(std::isalnum(static_cast<unsigned char>(expr[pos - 1])) || expr[pos - 1] == '_');
        const size_t end = pos + sym.size();
        const bool endOk = end >= expr.size() || !(std::isalnum(static_cast<unsigned char>(expr[end])) || expr[end] == '_');
        if (startOk && endOk) return true;
        pos = end;
    }
    return false;
}

}  // namespace

void HipGenericExecutor::hoistInits(const HipCodegen& cg, int first, int last,
                                    std::unordered_map<std::string, bool>& initDone,
                                    const std::unordered_map<std::string, const HipParamBinding*>& initSpec) {
    if (skipInit_) return;
    std::vector<void*> dst;
    std::vector<size_t> bytes;
    std::vector<const void*> pats;
    std::vector<int> plen;
    std::vector<std::vector<uint8_t>> periods;  // each buffer's pattern at its shortest period
    const auto& phases = cg.getPhases();
    for (int pi = first; pi < last; ++pi) {
        const auto& p = phases[static_cast<size_t>(pi)];
        for (const auto& b : p.bindings) {
            if (b.kind != HipParamKind::DeviceBuffer || initDone[b.name]) continue;
            auto sp = initSpec.find(b.name);
            if (sp == initSpec.end() || sp->second != &b) continue;  // not defined by this phase
            const HipParamBinding* ib = sp->second;
            bool late = false;
            for (const auto& sym : lateSymbols_) late |= mentionsSymbol(ib->sizeExpr, sym);
            if (late) continue;
            uint64_t elems = 0;
            try {
                elems = sizes_.resolve(ib->sizeExpr);
            } catch (const std::exception&) {
                continue;  // sized by something not known yet: initialised at its phase
            }
            size_t nb = static_cast<size_t>(elems) * ib->elemBytes;
            // zero fills may cover the allocation's padding (allocations are
            // whole 256-byte multiples), so byte arrays of any length join
            if (ib->init == InitKind::Zero) nb = (nb + 7) & ~static_cast<size_t>(7);
            periods.push_back(ib->init == InitKind::Zero ? std::vector<uint8_t>(8, 0) : shortestPeriod(ib->pattern));
            const int pl = static_cast<int>(periods.back().size());
            if (nb == 0 || !multiFillable(nb, pl)) {
                periods.pop_back();
                continue;
            }
            Buffer& buf = ensureBuffer(*ib);
            dst.push_back(buf.ptr);
            bytes.push_back(nb);
            plen.push_back(pl);
            initDone[b.name] = true;
        }
    }
    for (const auto& pp : periods) pats.push_back(pp.data());
    if (!dst.empty())
        check(gdb_fill_multi_async(static_cast<int>(dst.size()), dst.data(), bytes.data(), pats.data(), plen.data(),
                                   stream_),
              "gdb_fill_multi_async");
}

int HipGenericExecutor::occupancy(gdb_kernel k, int block) {
    auto key = std::make_pair(k, block);
    auto it = occupancy_.find(key);
    if (it != occupancy_.end()) return it->second;
    int nb = 1;
    if (gdb_kernel_occupancy(k, block, 0, &nb) != GDB_OK || nb < 1) nb = 1;
    occupancy_[key] = nb;
    return nb;
}

void HipGenericExecutor::prepare(const HipCodegen& cg, int firstPhase, int lastPhase) {
    const auto& phases = cg.getPhases();
    const int last = lastPhase < 0 ? static_cast<int>(phases.size()) : lastPhase;
    for (int pi = firstPhase; pi < last; ++pi) {
        for (const auto& b : phases[static_cast<size_t>(pi)].bindings) {
            if (b.kind != HipParamKind::DeviceBuffer) continue;
            try {
                ensureBuffer(b);
            } catch (const std::runtime_error&) {
                // Sized by a symbol a hook registers later; allocated at launch.
            }
        }
        resolveBufferTables();
    }
}

void HipGenericExecutor::launchPhase(RuntimeCompiler& rc, const RuntimeCompiler::CompiledQuery& cq,
                                     const HipCodegen::PhaseInfo& p, std::unordered_map<std::string, bool>& initDone,
                                     const std::unordered_map<std::string, const HipParamBinding*>& initSpec,
                                     bool foldFollows, unsigned* gridOut, gdb_event beforeKernel, bool* marked) {
    std::vector<uint64_t> args;
    args.reserve(p.bindings.size());
    bool filled = false;
    resolveBufferTables();
    for (const auto& b : p.bindings) {
        switch (b.kind) {
            case HipParamKind::TableColumn: {
                auto t = tables_.find(b.tableName);
                if (t == tables_.end()) throw std::runtime_error("executor: table '" + b.tableName + "' not registered");
                auto c = t->second.columns.find(b.columnName);
                if (c == t->second.columns.end())
                    throw std::runtime_error("executor: column '" + b.columnName + "' of table '" + b.tableName +
                                             "' not registered");
                args.push_back(reinterpret_cast<uint64_t>(c->second));
                break;
            }
            case HipParamKind::TableSize: {
                auto t = tables_.find(b.tableName);
                if (t == tables_.end()) throw std::runtime_error("executor: table '" + b.tableName + "' not registered");
                args.push_back(t->second.rows);
                break;
            }
            case HipParamKind::DeviceBuffer: {
                Buffer& buf = ensureBuffer(b);
                if (!skipInit_ && !initDone[b.name]) {
                    // A buffer is initialised right before the phase that
                    // defines it (the first phase binding it with an init
                    // kind), so a run over a phase range never re-fills a
                    // buffer an earlier phase built.
                    auto sp = initSpec.find(b.name);
                    const bool owner = sp != initSpec.end() && sp->second >= p.bindings.data() &&
                                       sp->second < p.bindings.data() + p.bindings.size();
                    if (owner) {
                        const HipParamBinding* ib = sp->second;
                        const size_t bytes = static_cast<size_t>(sizes_.resolve(ib->sizeExpr)) * ib->elemBytes;
                        if (ib->init == InitKind::Zero) {
                            const uint8_t z = 0;
                            check(gdb_fill_async(buf.ptr, bytes, &z, 1, stream_), "fill " + b.name);
                        } else {
                            check(gdb_fill_async(buf.ptr, bytes, ib->pattern.data(), static_cast<int>(ib->pattern.size()),
                                                 stream_),
                                  "fill " + b.name);
                        }
                        filled = true;
                        initDone[b.name] = true;
                    }
                }
                args.push_back(reinterpret_cast<uint64_t>(buf.ptr));
                break;
            }
            case HipParamKind::ScalarInt: {
                auto s = scalars_.find(b.name);
                if (s == scalars_.end()) throw std::runtime_error("executor: scalar '" + b.name + "' not registered");
                args.push_back(static_cast<uint64_t>(s->second));
                break;
            }
            case HipParamKind::SymbolValue:
                // partials that nothing folds would be missing from the result
                args.push_back(!foldFollows && b.name == p.partialsSymbol ? 0 : sizes_.resolve(b.sizeExpr));
                break;
        }
    }
    const int items = p.isSingleThread ? 1 : p.items;
    bool known = false;
    for (int v : (p.isSingleThread ? std::vector<int>{1} : p.itemsVariants)) known |= (v == items);
    if (!known) throw std::runtime_error("executor: phase " + p.name + " has no ITEMS=" + std::to_string(items) + " variant");
    const int block = p.isSingleThread ? 64 : p.threadgroupSize;
    if (block > p.launchBound && !p.isSingleThread)
        throw std::runtime_error("executor: block " + std::to_string(block) + " exceeds launch bound of " + p.name);
    gdb_kernel k = rc.getPipeline(cq, HipCodegen::kernelName(p.name, items));
    unsigned grid = 1;
    if (!p.isSingleThread) {
        const uint64_t rows = p.rowsExpr.empty() ? 1 : sizes_.resolve(p.rowsExpr);
        const uint64_t tile = static_cast<uint64_t>(block) * static_cast<uint64_t>(items);
        uint64_t need = std::max<uint64_t>(1, (rows + tile - 1) / tile);
        uint64_t cap = static_cast<uint64_t>(cuCount_) * static_cast<uint64_t>(occupancy(k, block));
        if (p.maxThreadgroups > 0) cap = std::min<uint64_t>(cap, static_cast<uint64_t>(p.maxThreadgroups));
        cap = std::max<uint64_t>(cap, 1);
        grid = static_cast<unsigned>(std::min(need, cap));
    }
    if (gridOut) *gridOut = grid;
    // A phase begins where the one before it ended unless something came
    // between (fills; *marked set by the caller: the start of the run, a hook):
    // a second event record between back-to-back kernels only cost time.
    if (beforeKernel && (filled || *marked)) {
        check(gdb_event_record(beforeKernel, stream_), "gdb_event_record");
        *marked = true;
    }
    check(gdb_launch(k, grid, static_cast<unsigned>(block), 0, args.data(), args.size() * 8, stream_),
          "launch " + p.name);
}

std::vector<uint64_t> HipGenericExecutor::packPhaseArgs(const HipCodegen& cg, int phase) {
    const auto& p = cg.getPhases().at(static_cast<size_t>(phase));
    resolveBufferTables();
    std::vector<uint64_t> args;
    for (const auto& b : p.bindings) {
        switch (b.kind) {
            case HipParamKind::TableColumn: {
                auto t = tables_.find(b.tableName);
                if (t == tables_.end()) throw std::runtime_error("executor: table '" + b.tableName + "' not registered");
                auto c = t->second.columns.find(b.columnName);
                if (c == t->second.columns.end())
                    throw std::runtime_error("executor: column '" + b.columnName + "' not registered");
                args.push_back(reinterpret_cast<uint64_t>(c->second));
                break;
            }
            case HipParamKind::TableSize: {
                auto t = tables_.find(b.tableName);
                if (t == tables_.end()) throw std::runtime_error("executor: table '" + b.tableName + "' not registered");
                args.push_back(t->second.rows);
                break;
            }
            case HipParamKind::DeviceBuffer: args.push_back(reinterpret_cast<uint64_t>(ensureBuffer(b).ptr)); break;
            case HipParamKind::ScalarInt: {
                auto s = scalars_.find(b.name);
                if (s == scalars_.end()) throw std::runtime_error("executor: scalar '" + b.name + "' not registered");
                args.push_back(static_cast<uint64_t>(s->second));
                break;
            }
            case HipParamKind::SymbolValue: args.push_back(sizes_.resolve(b.sizeExpr)); break;
        }
    }
    return args;
}

void HipGenericExecutor::collectInits(const HipCodegen& cg, FillList& out) {
    for (const auto& kv : initSpecs(cg)) {
        const HipParamBinding* ib = kv.second;
        Buffer& buf = ensureBuffer(*ib);
        size_t bytes = static_cast<size_t>(sizes_.resolve(ib->sizeExpr)) * ib->elemBytes;
        if (!bytes) continue;
        std::vector<uint8_t> pat = ib->init == InitKind::Zero ? std::vector<uint8_t>(8, 0) : shortestPeriod(ib->pattern);
        // zero fills may cover the allocation's padding (whole 256-byte multiples)
        if (ib->init == InitKind::Zero) bytes = (bytes + 7) & ~static_cast<size_t>(7);
        const int pl = static_cast<int>(pat.size());
        const bool multi = multiFillable(bytes, pl) && reinterpret_cast<uintptr_t>(buf.ptr) % 8 == 0 && bytes <= buf.bytes;
        if (!multi) {
            out.singles.push_back({buf.ptr, bytes, pat});
            continue;
        }
        std::array<uint8_t, 32> w{};
        for (int k = 0; k < 32; ++k) w[static_cast<size_t>(k)] = pat[static_cast<size_t>(k % pl)];
        out.dst.push_back(buf.ptr);
        out.bytes.push_back(bytes);
        out.pattern.push_back(w);
        out.plen.push_back(pl);
    }
}

std::vector<HipGenericExecutor::StatusRef> HipGenericExecutor::statusRefs(const HipCodegen& cg) const {
    std::vector<StatusRef> out;
    for (const auto& p : cg.getPhases()) {
        auto st = buffers_.find(p.statusBuffer);
        if (!p.statusBuffer.empty() && st != buffers_.end()) out.push_back({st->second.ptr, p.name, false, ""});
        auto ck = buffers_.find(p.checkBuffer);
        if (!p.checkBuffer.empty() && ck != buffers_.end()) out.push_back({ck->second.ptr, p.name, true, p.checkMessage});
    }
    return out;
}

void HipGenericExecutor::judgeStatus(const StatusRef& r, const uint64_t* w) {
    if (!r.check && w[0] != 0) throw GdbOverflowError(r.phase, w[2]);
    if (r.check && w[0] != 0)
        throw std::runtime_error("phase " + r.phase + ": " + r.message + " (" + std::to_string(w[2]) + " rows)");
}

void HipGenericExecutor::enqueueInits(const HipCodegen& cg) {
    for (const auto& kv : initSpecs(cg)) {
        const HipParamBinding* ib = kv.second;
        Buffer& buf = ensureBuffer(*ib);
        const size_t bytes = static_cast<size_t>(sizes_.resolve(ib->sizeExpr)) * ib->elemBytes;
        if (ib->init == InitKind::Zero) {
            const uint8_t z = 0;
            check(gdb_fill_async(buf.ptr, bytes, &z, 1, stream_), "fill " + ib->name);
        } else {
            check(gdb_fill_async(buf.ptr, bytes, ib->pattern.data(), static_cast<int>(ib->pattern.size()), stream_),
                  "fill " + ib->name);
        }
    }
}

void HipGenericExecutor::enqueue(RuntimeCompiler& rc, const RuntimeCompiler::CompiledQuery& cq, const HipCodegen& cg,
                                 int firstPhase, int lastPhase) {
    const auto& phases = cg.getPhases();
    const int last = lastPhase < 0 ? static_cast<int>(phases.size()) : lastPhase;
    auto spec = initSpecs(cg);
    std::unordered_map<std::string, bool> initDone;
    hoistInits(cg, firstPhase, last, initDone, spec);
    for (int pi = firstPhase; pi < last; ++pi)
        launchPhase(rc, cq, phases[static_cast<size_t>(pi)], initDone, spec, true, nullptr, nullptr, nullptr);
}

HipExecutionResult HipGenericExecutor::execute(RuntimeCompiler& rc, const RuntimeCompiler::CompiledQuery& cq,
                                               const HipCodegen& cg, int warmupRuns, int measuredRuns, int firstPhase,
                                               int lastPhase) {
    const auto& phases = cg.getPhases();
    const int last = lastPhase < 0 ? static_cast<int>(phases.size()) : lastPhase;
    const int np = last - firstPhase;
    HipExecutionResult res;
    auto t0 = std::chrono::steady_clock::now();
    prepare(cg, firstPhase, last);
    res.bufferAllocTimeMs =
        std::chrono::duration<float, std::milli>(std::chrono::steady_clock::now() - t0).count();
    while (static_cast<int>(events_.size()) < 2 * np + 1) {
        gdb_event e;
        check(gdb_event_create(&e), "gdb_event_create");
        events_.push_back(e);
    }
    auto spec = initSpecs(cg);
    const int runs = warmupRuns + std::max(1, measuredRuns);
    measuredPhase_.assign(static_cast<size_t>(np), 0.0f);
    measuredFill_.assign(static_cast<size_t>(np), 0.0f);
    PendingStatus pending;
    for (int r = 0; r < runs; ++r) {
        const bool measured = r >= warmupRuns;
        std::unordered_map<std::string, bool> initDone;
        res.phaseTimesMs.assign(static_cast<size_t>(np), 0.0f);
        res.phaseFillMs.assign(static_cast<size_t>(np), 0.0f);
        res.phaseNames.clear();
        res.phaseGrid.clear();
        res.phaseBlock.clear();
        res.phaseItems.clear();
        check(gdb_event_record(events_[0], stream_), "gdb_event_record");
        hoistInits(cg, firstPhase, last, initDone, spec);
        bool apart = true;  // something lies between the last event recorded and the next phase
        ownStart_.assign(static_cast<size_t>(np), true);
        for (int pi = firstPhase; pi < last; ++pi) {
            const auto& p = phases[static_cast<size_t>(pi)];
            unsigned grid = 0;
            const size_t e = static_cast<size_t>(2 * (pi - firstPhase));
            bool marked = apart;
            bool foldFollows = p.partialsSymbol.empty() || p.foldsPartials;
            for (int f = pi + 1; f < last && !foldFollows; ++f)
                foldFollows = phases[static_cast<size_t>(f)].partialsSymbol == p.partialsSymbol;
            launchPhase(rc, cq, p, initDone, spec, foldFollows, &grid, phaseTiming_ ? events_[e + 1] : nullptr, &marked);
            ownStart_[static_cast<size_t>(pi - firstPhase)] = marked;
            apart = false;
            if (phaseTiming_ || pi + 1 == last) check(gdb_event_record(events_[e + 2], stream_), "gdb_event_record");
            res.phaseNames.push_back(p.name);
            res.phaseGrid.push_back(grid);
            res.phaseBlock.push_back(static_cast<unsigned>(p.isSingleThread ? 64 : p.threadgroupSize));
            res.phaseItems.push_back(static_cast<unsigned>(p.isSingleThread ? 1 : p.items));
            auto h = hooks_.find(p.name);
            if (h != hooks_.end()) {
                if (h->second.bytes) {  // the hook's read rides behind the phase: one synchronisation
                    auto bit = buffers_.find(h->second.buffer);
                    if (bit == buffers_.end()) throw std::runtime_error("executor: no buffer " + h->second.buffer);
                    if (h->second.offset + h->second.bytes > bit->second.bytes)
                        throw std::runtime_error("executor: hook read past the end of " + h->second.buffer);
                    uint64_t* dst = ensurePinned(h->second.bytes);
                    check(gdb_memcpy_d2h_async(dst, static_cast<const char*>(bit->second.ptr) + h->second.offset,
                                               h->second.bytes, stream_),
                          "hook read " + h->second.buffer);
                }
                syncStream();
                h->second.fn(*this);
                apart = true;
            }
        }
        if (r + 1 == runs) {
            // the final run: status words gathered and read behind it, one wait for both
            pending = enqueueStatus(cg, firstPhase, last);
            syncStream();
        } else {
            check(gdb_event_sync(events_[static_cast<size_t>(2 * np)]), "gdb_event_sync");
        }
        if (measured) {
            const float w = 1.0f / static_cast<float>(std::max(1, measuredRuns));
            for (int i = 0; phaseTiming_ && i < np; ++i) {
                float ms = 0.0f, fill = 0.0f;
                const size_t e = static_cast<size_t>(2 * i);
                const bool own = ownStart_[static_cast<size_t>(i)];
                check(gdb_event_elapsed_ms(events_[own ? e + 1 : e], events_[e + 2], &ms), "gdb_event_elapsed_ms");
                if (own) check(gdb_event_elapsed_ms(events_[e], events_[e + 1], &fill), "gdb_event_elapsed_ms");
                measuredPhase_[static_cast<size_t>(i)] += ms * w;
                measuredFill_[static_cast<size_t>(i)] += fill * w;
            }
            float total = 0.0f;
            check(gdb_event_elapsed_ms(events_[0], events_[static_cast<size_t>(2 * np)], &total), "gdb_event_elapsed_ms");
            res.totalKernelTimeMs += total * w;
        }
    }
    res.phaseTimesMs = measuredPhase_;
    res.phaseFillMs = measuredFill_;
    res.phaseStatus = judgeStatuses(pending);
    return res;
}

HipGenericExecutor::PendingStatus HipGenericExecutor::enqueueStatus(const HipCodegen& cg, int firstPhase,
                                                                    int lastPhase) {
    // Every status and check word of the range is written to pinned memory by
    // one launch; the caller's next synchronisation covers it.
    const auto& phases = cg.getPhases();
    const int last = lastPhase < 0 ? static_cast<int>(phases.size()) : lastPhase;
    PendingStatus ps;
    ps.phases = static_cast<size_t>(std::max(0, last - firstPhase));
    std::vector<gdb_gather_piece> pieces;
    auto add = [&](int phase, void* words, const std::string& name, bool isCheck, const std::string& message) {
        pieces.push_back({words, 32u, static_cast<uint32_t>(32 * pieces.size())});
        ps.refs.push_back({phase, {words, name, isCheck, message}});
    };
    for (int pi = firstPhase; pi < last; ++pi) {
        const auto& p = phases[static_cast<size_t>(pi)];
        auto st = buffers_.find(p.statusBuffer);
        if (!p.statusBuffer.empty() && st != buffers_.end()) add(pi - firstPhase, st->second.ptr, p.name, false, "");
        auto ck = buffers_.find(p.checkBuffer);
        if (!p.checkBuffer.empty() && ck != buffers_.end())
            add(pi - firstPhase, ck->second.ptr, p.name, true, p.checkMessage);
    }
    if (ps.refs.empty()) return ps;
    uint64_t* host = ensurePinned(32 * pieces.size());
    for (size_t i = 0; i < pieces.size(); i += GDB_GATHER_MAX)
        check(gdb_gather_to_host(pieces.data() + i, static_cast<int>(std::min<size_t>(GDB_GATHER_MAX, pieces.size() - i)),
                                 host, stream_),
              "read status words");
    ps.host = host;
    return ps;
}

std::vector<std::array<uint64_t, 4>> HipGenericExecutor::judgeStatuses(const PendingStatus& ps) const {
    std::vector<std::array<uint64_t, 4>> out(ps.phases, {0, 0, 0, 0});
    for (size_t i = 0; i < ps.refs.size(); ++i) {
        const uint64_t* w = ps.host + 4 * i;
        judgeStatus(ps.refs[i].second, w);
        if (!ps.refs[i].second.check)
            for (int k = 0; k < 4; ++k) out[static_cast<size_t>(ps.refs[i].first)][static_cast<size_t>(k)] = w[k];
    }
    return out;
}

std::vector<std::array<uint64_t, 4>> HipGenericExecutor::checkStatus(const HipCodegen& cg, int firstPhase,
                                                                     int lastPhase) {
    const PendingStatus ps = enqueueStatus(cg, firstPhase, lastPhase);
    if (!ps.refs.empty()) syncStream();
    return judgeStatuses(ps);
}

void HipGenericExecutor::freeWorkspace(Workspace& w) {
    if (w.ptr) gdb_free(ctx_, w.ptr);  // waits for what still uses it
    w = Workspace{};
}

bool HipGenericExecutor::ensureWorkspace(Workspace& w, size_t bytes) {
    if (bytes <= w.bytes) return true;
    freeWorkspace(w);
    if (gdb_alloc(ctx_, bytes, &w.ptr) != GDB_OK) {
        w = Workspace{};
        return false;
    }
    w.bytes = bytes;
    return true;
}

std::shared_ptr<void> HipGenericExecutor::stagingFor(size_t bytes) {
    if (staging_ && staging_.use_count() == 1 && stagingBytes_ >= bytes) return staging_;
    if (bytes <= kKeepStaging) staging_.reset();
    void* h = nullptr;
    if (gdb_host_alloc_pinned(bytes, &h) != GDB_OK) return nullptr;
    std::shared_ptr<void> p(h, [](void* q) { gdb_host_free_pinned(q); });
    if (bytes <= kKeepStaging) {
        staging_ = p;
        stagingBytes_ = bytes;
    }
    return p;
}

namespace {
void groupColumns(const HipResultSchema& schema, GenericResult& res) {
    static const char* const names[4] = {"count", "sum", "min", "max"};
    res.columns.assign(5, ResultColumn{});
    res.columns[0].name = schema.hash.keyName;
    for (size_t k = 0; k < 4; ++k) res.columns[k + 1].name = names[k];
}
}  // namespace

const uint64_t* HipGenericExecutor::groupTable(const HipResultSchema& schema, uint64_t* slots) const {
    const auto& h = schema.hash;
    const auto it = buffers_.find(h.tableName);
    if (h.slotWords != 4 || it == buffers_.end()) return nullptr;
    *slots = sizes_.resolve(h.slotsSymbol);
    if (*slots > kMaxGroupSlots || *slots * 32 > it->second.bytes) return nullptr;
    return static_cast<const uint64_t*>(it->second.ptr);
}

// The columns of what gdb_group_rows_small wrote; false when it was too much.
bool HipGenericExecutor::smallGroups(const HipResultSchema& schema, const uint64_t* w, GenericResult& res) {
    const size_t n = static_cast<size_t>(w[0]);
    if (n > GDB_GROUP_ROWS_SMALL) return false;
    groupColumns(schema, res);
    const uint64_t* col = w + 8;
    for (auto& c : res.columns) c.i64.resize(n);
    for (size_t r = 0; r < n; ++r) {
        res.columns[0].i64[r] = static_cast<int64_t>(col[r] & 0xFFFFFFFFull);
        res.columns[1].i64[r] = static_cast<int64_t>(col[r] >> 32);
    }
    for (size_t k = 1; k < 4; ++k)
        if (n) std::memcpy(res.columns[k + 1].i64.data(), col + k * GDB_GROUP_ROWS_SMALL, n * 8);
    return true;
}

// The groups of a hash-aggregate table, ordered and split into columns on the
// device, so only the result crosses the link (32 bytes a group instead of 32
// a slot, from pinned memory) and the host sorts nothing. A group-by of 40M
// rows with 2.2M groups in 8M slots took 392 ms with the table copied and
// sorted on the host, 4.9 ms so; 8M rows with 400K groups 82 and 1.4 ms.
// Tables of at most 2 * GDB_GROUP_ROWS_SMALL slots take one launch of one
// block that writes the rows to pinned memory itself; a larger one would keep
// that block busy longer than the general path's dozen launches take. False
// when the workspace cannot be had (the caller reads the table instead).
bool HipGenericExecutor::collectGroups(const HipResultSchema& schema, GenericResult& res) {
    uint64_t slots = 0;
    const uint64_t* table = groupTable(schema, &slots);
    if (!table) return false;
    if (slots <= 2 * GDB_GROUP_ROWS_SMALL) {
        auto out = stagingFor(GDB_GROUP_ROWS_SMALL_BYTES);
        if (!out) return false;
        uint64_t* w = static_cast<uint64_t*>(out.get());
        check(gdb_group_rows_small(table, slots, w, stream_), "gdb_group_rows_small");
        syncStream();
        if (smallGroups(schema, w, res)) return true;
    }
    groupColumns(schema, res);

    // workspaces: head | pairs; once the number of groups is known, sort scratch | columns
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    if (!ensureWorkspace(groupPairs_, 256 + static_cast<size_t>(slots) * 8)) return false;
    uint64_t* const head = static_cast<uint64_t*>(groupPairs_.ptr);
    uint64_t* const pairs = head + 32;
    uint64_t* host = ensurePinned(16);
    check(gdb_group_rows_compact(table, slots, pairs, head, stream_), "gdb_group_rows_compact");
    check(gdb_memcpy_d2h_async(host, head, 16, stream_), "read group count");
    syncStream();
    const uint64_t n = host[0], maxKey = host[1];
    if (n == 0) return true;
    const size_t col8 = up(static_cast<size_t>(n) * 8), col4 = up(static_cast<size_t>(n) * 4);
    const size_t scratch = up(gdb_group_rows_scratch_bytes(n)), colBytes = 3 * col8 + 2 * col4;
    if (!ensureWorkspace(groupCols_, scratch + colBytes)) return false;
    auto out = stagingFor(colBytes);
    if (!out) return false;
    char* const cols = static_cast<char*>(groupCols_.ptr) + scratch;
    const size_t at[5] = {3 * col8, 3 * col8 + col4, 0, col8, 2 * col8};  // key, count, sum, min, max
    check(gdb_group_rows_sort(table, pairs, n, maxKey, groupCols_.ptr, reinterpret_cast<uint32_t*>(cols + at[0]),
                              reinterpret_cast<uint32_t*>(cols + at[1]), reinterpret_cast<int64_t*>(cols + at[2]),
                              reinterpret_cast<int64_t*>(cols + at[3]), reinterpret_cast<int64_t*>(cols + at[4]), stream_),
          "gdb_group_rows_sort");
    check(gdb_memcpy_d2h_async(out.get(), cols, colBytes, stream_), "read group columns");
    syncStream();
    for (size_t k = 0; k < 5; ++k) {
        auto& c = res.columns[k];
        c.hold = out;
        c.raw = static_cast<const char*>(out.get()) + at[k];
        c.raw32 = k < 2;
        c.rawRows = static_cast<size_t>(n);
    }
    if (groupPairs_.bytes > kKeepWorkspace) freeWorkspace(groupPairs_);
    if (groupCols_.bytes > kKeepWorkspace) freeWorkspace(groupCols_);
    return true;
}

GenericResult HipGenericExecutor::collectResult(const HipCodegen& cg) {
    if (cg.getResultSchema().kind == HipResultSchema::HASH_AGG) {
        GenericResult res;
        if (collectGroups(cg.getResultSchema(), res)) return res;
    }
    // The few words of a small result are written to pinned memory by one
    // launch and one wait serves them all; the collector's reads are answered
    // from there, or by a copy when they go beyond (more rows than the piece).
    size_t total = 0;
    const auto have = resultPieces(cg.getResultSchema(), &total);
    const char* host = nullptr;
    if (!have.empty()) {
        uint64_t* pinned = ensurePinned(total);
        host = reinterpret_cast<const char*>(pinned);
        std::vector<gdb_gather_piece> pieces;
        for (const auto& h : have)
            pieces.push_back({buffers_.at(h.name).ptr, static_cast<uint32_t>(h.bytes), static_cast<uint32_t>(h.at)});
        check(gdb_gather_to_host(pieces.data(), static_cast<int>(pieces.size()), pinned, stream_), "read result");
    }
    syncStream();
    return collectPieces(cg.getResultSchema(), have, host);
}

std::vector<HipGenericExecutor::Piece> HipGenericExecutor::resultPieces(const HipResultSchema& schema,
                                                                        size_t* total) const {
    std::vector<Piece> have;
    for (const auto& b : resultBuffers(schema)) {
        auto it = buffers_.find(b.name);
        if (it == buffers_.end()) continue;
        if (b.whole && b.bytes > kMaxPiece) continue;  // one read, of more than the piece could hold
        const size_t bytes = std::min({b.bytes, it->second.bytes, kMaxPiece}) / 4 * 4;
        if (bytes == 0) continue;
        have.push_back({b.name, bytes, *total});
        *total += (bytes + 15) / 16 * 16;
    }
    return have;
}

GenericResult HipGenericExecutor::collectPieces(const HipResultSchema& schema, const std::vector<Piece>& have,
                                                const char* host) {
    return HipResultCollector::collect(
        schema,
        [&](const std::string& name, size_t off, void* dst, size_t bytes) {
            for (const auto& h : have)
                if (h.name == name && off + bytes <= h.bytes) {
                    std::memcpy(dst, host + h.at + off, bytes);
                    return;
                }
            readBuffer(name, off, dst, bytes);
        },
        [this](const std::string& expr) { return sizes_.resolve(expr); });
}

// A batch of 64 pipelines whose results were read one by one spent 34 us on
// each, most of it a launch and a wait: with one launch for the 32 group
// tables, one for the others' words and one wait, replay and results take
// 1.09 ms instead of 2.64. A result with more than kPieces bytes to read, another
// context or stream than the first runner's, or too many groups is collected
// by itself afterwards (the shared pinned block is free again then).
std::vector<GenericResult> HipGenericExecutor::collectMany(
    const std::vector<std::pair<HipGenericExecutor*, const HipCodegen*>>& runs) {
    constexpr size_t kPieces = 1024;
    std::vector<GenericResult> res(runs.size());
    if (runs.empty()) return res;
    HipGenericExecutor& first = *runs[0].first;
    enum Way { ALONE, GROUPS, PIECES };
    std::vector<Way> way(runs.size(), ALONE);
    std::vector<std::shared_ptr<void>> staged(runs.size());
    std::vector<std::vector<Piece>> have(runs.size());
    std::vector<gdb_group_table> tables;
    std::vector<gdb_gather_piece> pieces;
    size_t total = 0;
    for (size_t i = 0; i < runs.size(); ++i) {
        HipGenericExecutor& ex = *runs[i].first;
        const HipResultSchema& schema = runs[i].second->getResultSchema();
        if (ex.ctx_ != first.ctx_ || ex.stream_ != first.stream_) continue;
        if (schema.kind == HipResultSchema::HASH_AGG) {
            uint64_t slots = 0;
            const uint64_t* table = ex.groupTable(schema, &slots);
            if (!table || slots > 2 * GDB_GROUP_ROWS_SMALL) continue;
            staged[i] = ex.stagingFor(GDB_GROUP_ROWS_SMALL_BYTES);
            if (!staged[i]) continue;
            tables.push_back({table, static_cast<uint64_t*>(staged[i].get()), slots});
            way[i] = GROUPS;
            continue;
        }
        size_t bytes = 0;
        auto own = ex.resultPieces(schema, &bytes);
        if (own.empty() || bytes > kPieces) continue;
        for (auto& h : own) {
            h.at += total;
            pieces.push_back({ex.buffers_.at(h.name).ptr, static_cast<uint32_t>(h.bytes), static_cast<uint32_t>(h.at)});
        }
        total += bytes;
        have[i] = std::move(own);
        way[i] = PIECES;
    }
    const char* host = nullptr;
    if (!tables.empty())
        check(gdb_group_rows_small_many(tables.data(), static_cast<int>(tables.size()), first.stream_),
              "gdb_group_rows_small_many");
    if (!pieces.empty()) {
        uint64_t* pinned = first.ensurePinned(total);
        host = reinterpret_cast<const char*>(pinned);
        for (size_t at = 0; at < pieces.size(); at += GDB_GATHER_MAX)
            check(gdb_gather_to_host(pieces.data() + at,
                                     static_cast<int>(std::min<size_t>(GDB_GATHER_MAX, pieces.size() - at)), pinned,
                                     first.stream_),
                  "read results");
    }
    if (!tables.empty() || !pieces.empty()) first.syncStream();
    for (size_t i = 0; i < runs.size(); ++i) {
        const HipResultSchema& schema = runs[i].second->getResultSchema();
        if (way[i] == PIECES)
            res[i] = runs[i].first->collectPieces(schema, have[i], host);
        else if (way[i] == GROUPS && !smallGroups(schema, static_cast<uint64_t*>(staged[i].get()), res[i]))
            way[i] = ALONE;
        staged[i].reset();
    }
    for (size_t i = 0; i < runs.size(); ++i)
        if (way[i] == ALONE) res[i] = runs[i].first->collectResult(*runs[i].second);
    return res;
}

std::vector<HipGenericExecutor::ResultRead> HipGenericExecutor::resultBuffers(const HipResultSchema& rs) const {
    switch (rs.kind) {
        case HipResultSchema::KEYED_AGG:
            return {{rs.keyed.bufferName, static_cast<size_t>(rs.keyed.numBuckets) * static_cast<size_t>(rs.keyed.wordsPerBucket) * 8, true}};
        case HipResultSchema::TOPK:
            return {{rs.topk.ctlBuffer, 32, true}, {rs.topk.bufferName, 16 * static_cast<size_t>(rs.topk.k), true}};
        case HipResultSchema::HISTOGRAM:
        case HipResultSchema::COUNTS:
            return {{rs.counts.bufferName, static_cast<size_t>(sizes_.resolve(rs.counts.sizeExpr)) * 4, true}};
        case HipResultSchema::ROWS:
            return {{rs.rows.ctlBuffer, 32, true}, {rs.rows.bufferName, rs.rows.fields.size() * 8 * 64, false}};  // the first 64 rows
        default: return {};
    }
}

void HipGenericExecutor::releaseAllocatedBuffers() {
    for (auto& kv : buffers_)
        if (kv.second.owned && kv.second.ptr) gdb_free(ctx_, kv.second.ptr);
    buffers_.clear();
    freeWorkspace(groupPairs_);
    freeWorkspace(groupCols_);
    staging_.reset();
    stagingBytes_ = 0;
}

void* HipGenericExecutor::getAllocatedBuffer(const std::string& name) const {
    auto it = buffers_.find(name);
    return it == buffers_.end() ? nullptr : it->second.ptr;
}

size_t HipGenericExecutor::getAllocatedBytes(const std::string& name) const {
    auto it = buffers_.find(name);
    return it == buffers_.end() ? 0 : it->second.bytes;
}

size_t HipGenericExecutor::ownedBytes() const {
    size_t n = groupPairs_.bytes + groupCols_.bytes;
    for (const auto& kv : buffers_)
        if (kv.second.owned) n += kv.second.bytes;
    return n;
}

void HipGenericExecutor::readBuffer(const std::string& name, size_t offset, void* host, size_t bytes) const {
    auto it = buffers_.find(name);
    if (it == buffers_.end()) throw std::runtime_error("executor: no buffer " + name);
    if (offset + bytes > it->second.bytes)
        throw std::runtime_error("executor: read past the end of buffer " + name);
    check(gdb_memcpy_d2h_async(host, static_cast<const char*>(it->second.ptr) + offset, bytes, stream_),
          "read " + name);
    check(gdb_stream_sync(stream_), "gdb_stream_sync");
}

}  // namespace codegen
}  // namespace gdb
