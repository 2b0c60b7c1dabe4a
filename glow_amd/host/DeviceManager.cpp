#include "DeviceManager.h"

#include "glow_mi355x.h"

#include <algorithm>
#include <cstring>
#include <future>

namespace glow_mi355x {

namespace {
// Bounds of the pinned memory a device manager keeps for its requests. Inputs that
// do not fit together go through it in turns; a single tensor larger than it, and
// outputs beyond theirs, are copied by the runtime.
constexpr size_t kStagingLeast = 1 << 20, kStagingMost = 64 << 20, kOutputsMost = 4 << 20;
// Pinned inputs of at least this size that need no other form on the device are
// copied by the DMA engines, whose set-up is small against them, without the CPU.
constexpr size_t kDirectCopy = 1 << 20;
// Staged bytes per copy of an input that no launch waits for.
constexpr size_t kLateCopy = 4 << 20;
// A float input that the network quantizes first is quantized while it is staged:
// a quarter of the bytes over PCIe. Two helper threads are what it takes to do that
// faster than the link moves the floats (38.5 MB: 0.69 ms by DMA; quantized by one
// thread 1.0 ms, by four 0.27 and pulled meanwhile).
constexpr int kQuantizeHelpers = 2;
// Launches issued one by one serve a function when they took at most this share of the
// fastest recording's time: the host is at work for as long as it issues them (2.5 us each),
// for one replay of a graph no longer than 24 us.
constexpr float kDirectShare = 0.97f;
// Room for a function's quantized inputs behind its generated constants.
size_t quantizedBytes(const MI355XFunction &fn) {
  return fn.quantizedBytes ? fn.quantizedBytes + 256 : 0;
}
// Whether any lookup of `fn` takes its bag positions from placeholder `name`.
bool derivesFrom(const MI355XFunction &fn, const std::string &name) {
  for (const auto &d : fn.derivedBagOffsets)
    if (d.lengths == name) return true;
  return false;
}
// Whether `fn` takes an input quantized that `writer` writes on the device.
bool quantizesWhatIsWritten(const MI355XFunction &fn, const MI355XFunction &writer) {
  for (const auto &q : fn.quantizedInputs)
    for (const auto &w : writer.writtenPlaceholders)
      if (q.placeholder == w) return true;
  return false;
}
} // namespace

namespace {
Error fromStatus(int rc, const char *what) {
  if (rc == MI355X_OK) return Error::success();
  ErrorCode c = ErrorCode::RUNTIME_ERROR;
  if (rc == MI355X_ERR_OUT_OF_DEVICE_MEMORY) c = ErrorCode::RUNTIME_OUT_OF_DEVICE_MEMORY;
  else if (rc == MI355X_ERR_NOT_SUPPORTED) c = ErrorCode::DEVICE_FEATURE_NOT_SUPPORTED;
  else if (rc == MI355X_ERR_DEVICE_NOT_FOUND) c = ErrorCode::RUNTIME_DEVICE_NOT_FOUND;
  return MI355X_MAKE_ERR(c, "%s: %s", what, mi355x_last_error());
}
} // namespace

MI355XDeviceManager::~MI355XDeviceManager() { (void)stop(true); }

void MI355XDeviceManager::enqueue(std::function<void()> work) {
  {
    std::lock_guard<std::mutex> lk(mu_);
    queue_.push_back(std::move(work));
  }
  cv_.notify_one();
}

void MI355XDeviceManager::workerLoop() {
  for (;;) {
    std::function<void()> work;
    {
      std::unique_lock<std::mutex> lk(mu_);
      cv_.wait(lk, [this] { return !busy_ && (stopping_ || !queue_.empty()); });
      if (queue_.empty()) return; // stopping and drained
      work = std::move(queue_.front());
      queue_.pop_front();
      busy_ = true;
    }
    work();
    std::lock_guard<std::mutex> lk(mu_);
    busy_ = false;
  }
}

Error MI355XDeviceManager::init() {
  {
    std::lock_guard<std::mutex> lk(mu_);
    if (running_) return Error::success();
    running_ = true;
    stopping_ = false;
  }
  worker_ = std::thread([this] { workerLoop(); });
  // the device is bound to the worker thread, so bind it there
  std::promise<Error> done;
  auto fut = done.get_future();
  enqueue([this, &done] {
    int n = 0;
    if (mi355x_num_devices(&n) != MI355X_OK || config_.deviceID < 0 || config_.deviceID >= n) {
      done.set_value(MI355X_MAKE_ERR(ErrorCode::RUNTIME_DEVICE_NOT_FOUND,
                                     "no MI355X device %d (%d visible)", config_.deviceID, n));
      return;
    }
    int rc = mi355x_init(config_.deviceID);
    if (rc != MI355X_OK) {
      done.set_value(MI355X_MAKE_ERR(ErrorCode::RUNTIME_DEVICE_NOT_FOUND, "%s", mi355x_last_error()));
      return;
    }
    mi355x_info info;
    rc = mi355x_device_info(&info);
    if (rc == MI355X_OK) rc = mi355x_stream_create(&stream_);
    if (rc == MI355X_OK) rc = mi355x_stream_create(&lateStream_);
    for (int i = 1; i < config_.graphBranches && rc == MI355X_OK; i++) {
      void *s = nullptr;
      rc = mi355x_stream_create(&s);
      if (rc == MI355X_OK) sideStreams_.push_back(s);
    }
    if (rc == MI355X_OK) rc = mi355x_host_alloc((void **)&done_, 64);
    if (rc == MI355X_OK) rc = mi355x_malloc((void **)&arrived_, 64);
    if (rc == MI355X_OK) {
      *done_ = doneValue_ = 0;
      rc = mi355x_fill_u8(arrived_, 0, 64, stream_);
    }
    if (rc == MI355X_OK) rc = mi355x_stream_sync(stream_);
    if (rc != MI355X_OK) {
      done.set_value(fromStatus(rc, "device set-up"));
      return;
    }
    pool_.reset(new StagingPool());
    info_.name = info.name;
    info_.arch = info.arch;
    info_.totalMemory = info.total_memory;
    info_.computeUnits = info.compute_units;
    maxMemoryBytes_ = config_.deviceMemory ? config_.deviceMemory : info.free_memory;
    done.set_value(Error::success());
  });
  Error e = fut.get();
  if (e) (void)stop(true);
  return e;
}

Error MI355XDeviceManager::stop(bool block) {
  (void)block;
  {
    std::lock_guard<std::mutex> lk(mu_);
    if (!running_) return Error::success();
  }
  std::promise<void> done;
  auto fut = done.get_future();
  enqueue([this, &done] {
    for (auto &kv : functions_) release(kv.second);
    functions_.clear();
    for (auto &kv : modules_)
      if (kv.second.arena) mi355x_arena_destroy(kv.second.arena);
    modules_.clear();
    usedMemoryBytes_ = 0;
    if (stream_) {
      mi355x_stream_sync(stream_);
      mi355x_stream_destroy(stream_);
      stream_ = nullptr;
    }
    for (void *s : sideStreams_) mi355x_stream_destroy(s);
    sideStreams_.clear();
    if (lateStream_) mi355x_stream_destroy(lateStream_);
    lateStream_ = nullptr;
    pool_.reset();
    mi355x_host_free(staging_);
    mi355x_host_free(outputs_);
    mi355x_host_free(done_);
    mi355x_free(arrived_);
    staging_ = outputs_ = nullptr;
    stagingBytes_ = 0;
    done_ = arrived_ = nullptr;
    done.set_value();
  });
  fut.get();
  {
    std::lock_guard<std::mutex> lk(mu_);
    stopping_ = true;
  }
  cv_.notify_all();
  if (worker_.joinable()) worker_.join();
  {
    std::lock_guard<std::mutex> lk(mu_);
    running_ = false;
  }
  return Error::success();
}

void MI355XDeviceManager::addNetwork(const Module *module, FunctionMapTy functions,
                                     ReadyCBTy readyCB) {
  {
    std::lock_guard<std::mutex> lk(mu_);
    if (!running_ || stopping_) {
      readyCB(module, MI355X_MAKE_ERR(ErrorCode::RUNTIME_REQUEST_REFUSED,
                                      "device manager is not running"));
      return;
    }
  }
  enqueue([this, module, functions, readyCB]() mutable {
    addNetworkImpl(module, std::move(functions), std::move(readyCB));
  });
}

void MI355XDeviceManager::evictNetwork(std::string functionName, EvictFunctionCBTy evictCB) {
  {
    std::lock_guard<std::mutex> lk(mu_);
    if (!running_ || stopping_) {
      evictCB(functionName, MI355X_MAKE_ERR(ErrorCode::RUNTIME_REQUEST_REFUSED,
                                            "device manager is not running"));
      return;
    }
  }
  enqueue([this, functionName, evictCB]() mutable {
    evictNetworkImpl(std::move(functionName), std::move(evictCB));
  });
}

RunIdentifierTy MI355XDeviceManager::runFunction(std::string functionName,
                                                 std::unique_ptr<ExecutionContext> ctx,
                                                 ResultCBTy resultCB) {
  const RunIdentifierTy id = nextRun_++;
  {
    std::lock_guard<std::mutex> lk(mu_);
    if (!running_ || stopping_) {
      resultCB(id, MI355X_MAKE_ERR(ErrorCode::RUNTIME_REQUEST_REFUSED,
                                   "device manager is not running"),
               std::move(ctx));
      return id;
    }
  }
  // std::function needs copyable captures: hand the context over by raw pointer
  ExecutionContext *raw = ctx.release();
  enqueue([this, id, functionName, raw, resultCB]() mutable {
    std::unique_ptr<ExecutionContext> ctx(raw);
    if (!ctx) {
      resultCB(id, MI355X_MAKE_ERR(ErrorCode::RUNTIME_ERROR, "no execution context"), nullptr);
      return;
    }
    std::vector<BoundArray> arrays;
    for (const auto &kv : ctx->getPlaceholderBindings()->pairs())
      if (kv.second) arrays.push_back({kv.first.c_str(), kv.second->data(), kv.second->sizeInBytes()});
    Error e = runRequest(functionName, arrays.data(), arrays.size());
    resultCB(id, std::move(e), std::move(ctx));
  });
  return id;
}

Error MI355XDeviceManager::runFunctionBlocking(const char *functionName, const BoundArray *arrays,
                                               size_t n) {
  bool here = false;
  {
    std::lock_guard<std::mutex> lk(mu_);
    if (!running_ || stopping_)
      return MI355X_MAKE_ERR(ErrorCode::RUNTIME_REQUEST_REFUSED, "device manager is not running");
    if (!busy_ && queue_.empty()) here = busy_ = true;
  }
  if (here) {
    int before = config_.deviceID;
    int rc = mi355x_set_device(config_.deviceID, &before);
    Error e = rc == MI355X_OK ? runRequest(functionName, arrays, n) : fromStatus(rc, "device");
    if (before != config_.deviceID) mi355x_set_device(before, nullptr);
    bool waiting;
    {
      std::lock_guard<std::mutex> lk(mu_);
      busy_ = false;
      waiting = stopping_ || !queue_.empty();
    }
    if (waiting) cv_.notify_one();
    return e;
  }
  std::promise<Error> p;
  auto fut = p.get_future();
  enqueue([&] { p.set_value(runRequest(functionName, arrays, n)); });
  return fut.get();
}

void MI355XDeviceManager::transferStaticPlaceholderToDevice(
    const Module *module, std::string placeholderName, Tensor *tensor,
    std::function<void(Error)> resultCB) {
  {
    std::lock_guard<std::mutex> lk(mu_);
    if (!running_ || stopping_) {
      resultCB(MI355X_MAKE_ERR(ErrorCode::RUNTIME_REQUEST_REFUSED, "device manager is not running"));
      return;
    }
  }
  enqueue([this, module, placeholderName, tensor, resultCB] {
    auto mit = modules_.find(module);
    if (!module || mit == modules_.end() || !mit->second.arena || !tensor) {
      resultCB(MI355X_MAKE_ERR(ErrorCode::RUNTIME_ERROR,
                               "cannot copy placeholder %s: its module has no function on this device",
                               placeholderName.c_str()));
      return;
    }
    const int id = module->getValueByName(placeholderName);
    if (id < 0 || module->value(id).category != SymbolCategory::Placeholder) {
      resultCB(MI355X_MAKE_ERR(ErrorCode::RUNTIME_ERROR, "%s is not a placeholder of the module",
                               placeholderName.c_str()));
      return;
    }
    const Value &v = module->value(id);
    if (tensor->sizeInBytes() > v.type.sizeInBytes()) {
      resultCB(MI355X_MAKE_ERR(ErrorCode::RUNTIME_ERROR, "tensor for %s has %zu bytes, slot %zu",
                               placeholderName.c_str(), tensor->sizeInBytes(), v.type.sizeInBytes()));
      return;
    }
    int rc = mi355x_arena_upload(mit->second.arena, MI355X_REGION_MUTABLE, v.offset, tensor->data(),
                                 tensor->sizeInBytes(), stream_);
    // lookups of the module's functions that take their bags from this placeholder
    if (rc == MI355X_OK) {
      for (auto &f : functions_) {
        if (f.second.module != module) continue;
        auto it = f.second.slots.find(placeholderName);
        if (it == f.second.slots.end()) continue;   // (the same in every function that has it)
        const Slot &s = it->second;
        rc = lengthsInSlot(s.derived, s.device, s.bytes, tensor->sizeInBytes());
        if (rc == MI355X_OK) rc = quantizeSlot(s.quantized, s.device, tensor->sizeInBytes());
        if (rc == MI355X_OK) rc = refreshOverlapped(s);
        break;
      }
    }
    if (rc == MI355X_OK) rc = mi355x_stream_sync(stream_);
    resultCB(rc == MI355X_OK ? Error::success() : fromStatus(rc, "placeholder copy"));
  });
}

Expected<float> MI355XDeviceManager::timeFunction(const std::string &functionName, int iterations) {
  {
    std::lock_guard<std::mutex> lk(mu_);
    if (!running_ || stopping_)
      return MI355X_MAKE_ERR(ErrorCode::RUNTIME_REQUEST_REFUSED, "device manager is not running");
  }
  if (iterations < 1)
    return MI355X_MAKE_ERR(ErrorCode::RUNTIME_ERROR, "iterations must be positive");
  std::promise<std::pair<Error, float>> done;
  auto fut = done.get_future();
  enqueue([this, &done, functionName, iterations] {
    auto it = functions_.find(functionName);
    if (it == functions_.end()) {
      done.set_value({MI355X_MAKE_ERR(ErrorCode::RUNTIME_NET_NOT_FOUND, "Function %s not found",
                                      functionName.c_str()),
                      0.0f});
      return;
    }
    FunctionResident &fr = it->second;
    ExecutionContext ctx;
    ctx.setDeviceBindings(std::unique_ptr<DeviceBindings>(new DeviceBindings(fr.bindings)));
    void *e0 = nullptr, *e1 = nullptr;
    Error err;
    float ms = 0.0f;
    // the comparison of recordings, if still going on, finishes untimed
    while (!fr.branchesTuned && !err) err = executeTuned(fr, &ctx);
    int rc = mi355x_event_create(&e0);
    if (rc == MI355X_OK) rc = mi355x_event_create(&e1);
    if (rc == MI355X_OK) rc = mi355x_stream_sync(stream_);
    if (rc == MI355X_OK) rc = mi355x_event_record(e0, stream_);
    if (rc != MI355X_OK && !err) err = fromStatus(rc, "timing set-up");
    for (int i = 0; i < iterations && !err; i++) err = fr.fn->execute(&ctx);
    if (!err) {
      rc = mi355x_event_record(e1, stream_);
      if (rc == MI355X_OK) rc = mi355x_event_sync(e1);
      if (rc == MI355X_OK) rc = mi355x_event_elapsed_ms(e0, e1, &ms);
      if (rc != MI355X_OK) err = fromStatus(rc, "timing");
    }
    mi355x_stream_sync(stream_);
    if (e0) mi355x_event_destroy(e0);
    if (e1) mi355x_event_destroy(e1);
    done.set_value({std::move(err), ms / (float)iterations});
  });
  auto r = fut.get();
  if (r.first) return r.first;
  return r.second;
}

Expected<int> MI355XDeviceManager::recordedBranches(const std::string &functionName) {
  {
    std::lock_guard<std::mutex> lk(mu_);
    if (!running_ || stopping_)
      return MI355X_MAKE_ERR(ErrorCode::RUNTIME_REQUEST_REFUSED, "device manager is not running");
  }
  std::promise<int> done;
  auto fut = done.get_future();
  enqueue([this, &done, functionName] {
    auto it = functions_.find(functionName);
    done.set_value(it == functions_.end() ? -1 : it->second.fn->recordedBranches(it->second.bindings));
  });
  const int branches = fut.get();
  if (branches < 0)
    return MI355X_MAKE_ERR(ErrorCode::RUNTIME_NET_NOT_FOUND, "Function %s not found",
                           functionName.c_str());
  return branches;
}

void MI355XDeviceManager::release(FunctionResident &fr) {
  if (fr.fn) fr.fn->dropGraph(fr.bindings);
  if (fr.arena) mi355x_arena_destroy(fr.arena);
  fr.arena = nullptr;
  usedMemoryBytes_ -= fr.bytes;
  auto it = modules_.find(fr.module);
  if (it != modules_.end() && --it->second.users == 0) {
    if (it->second.arena) mi355x_arena_destroy(it->second.arena);
    usedMemoryBytes_ -= it->second.bytes;
    modules_.erase(it);
  }
}

// `bytes` of a lengths placeholder have just been copied into its slot (slotBytes
// long). If lookups take their bag positions from it, the rest of the slot is
// cleared (a partial tensor: the missing bags are empty for the kernels that read
// the lengths and for the positions alike) and the positions are summed.
int MI355XDeviceManager::lengthsInSlot(const std::vector<DerivedPositions> &derived, uint8_t *slot,
                                       size_t slotBytes, size_t bytes) {
  if (derived.empty()) return MI355X_OK;
  int rc = MI355X_OK;
  if (bytes < slotBytes) rc = mi355x_fill_u8(slot + bytes, 0, slotBytes - bytes, stream_);
  for (const auto &d : derived) {
    if (rc != MI355X_OK) break;
    const mi355x_copy_segment s{nullptr,     slot, d.bags * sizeof(int32_t),
                                d.positions, (uint32_t)d.bags, MI355X_SEGMENT_LENGTHS};
    rc = mi355x_copy_segments(&s, 1, nullptr, 0, nullptr, stream_);
  }
  return rc;
}

// The quantized copies of a float placeholder, from the first `bytes` of its slot.
int MI355XDeviceManager::quantizeSlot(const std::vector<QuantizedCopy> &copies, const uint8_t *slot,
                                      size_t bytes) {
  int rc = MI355X_OK;
  for (const auto &q : copies)
    if (rc == MI355X_OK)
      rc = mi355x_quantize_i8(q.values, (const float *)slot, std::min(q.elements, (bytes + 3) / 4),
                              q.scale, q.offset, stream_);
  return rc;
}

int MI355XDeviceManager::refreshOverlapped(const Slot &s) {
  int rc = MI355X_OK;
  for (const Slot *o : s.overlapped) {
    if (rc == MI355X_OK) rc = lengthsInSlot(o->derived, o->device, o->bytes, o->bytes);
    if (rc == MI355X_OK) rc = quantizeSlot(o->quantized, o->device, o->bytes);
  }
  return rc;
}

// The slots of every resident function of `module`, after its set of functions has
// changed: the bag positions that follow a lengths placeholder belong to the
// module, so a request to one function refreshes those of all of them.
void MI355XDeviceManager::bindSlots(const Module *module) {
  for (auto &f : functions_) {
    FunctionResident &fr = f.second;
    if (fr.module != module) continue;
    fr.slots.clear();
    for (const auto &kv : fr.fn->getRuntimeBundle().symbolTable) {
      if (kv.second.symbolCategory != SymbolCategory::Placeholder) continue;
      Slot s;
      s.device = fr.bindings.mutableMem + kv.second.offset;
      s.bytes = kv.second.size;
      s.input = kv.second.input;
      s.output = kv.second.output;
      s.indices64 = kv.second.type.kind == ElemKind::Int64ITy;
      for (auto &g : functions_)
        if (g.second.module == module)
          for (const auto &d : g.second.fn->derivedBagOffsets)
            if (d.lengths == kv.first)
              s.derived.push_back({(int32_t *)d.ptr(g.second.bindings), d.segments});
      s.floatRead = false;
      for (auto &g : functions_) {
        if (g.second.module != module) continue;
        auto st = g.second.fn->getRuntimeBundle().symbolTable.find(kv.first);
        if (st == g.second.fn->getRuntimeBundle().symbolTable.end()) continue;
        bool sole = false;
        for (size_t i = 0; i < g.second.quantized.size(); i++)
          if (g.second.fn->quantizedInputs[i].placeholder == kv.first) {
            s.quantized.push_back(g.second.quantized[i]);
            sole = g.second.fn->quantizedInputs[i].sole;
          }
        if ((st->second.input && !sole) || st->second.output) s.floatRead = true;
      }
      fr.slots.emplace(kv.first, std::move(s));
    }
    for (auto &a : fr.slots) {
      Slot &s = a.second;
      for (const auto &b : fr.slots) {
        const Slot &o = b.second;
        if (&o != &s && !(o.derived.empty() && o.quantized.empty()) && o.device < s.device + s.bytes &&
            s.device < o.device + o.bytes)
          s.overlapped.push_back(&o);
      }
    }
  }
}

// Room for inputs of `bytes` in all, within the bound; never shrinks.
int MI355XDeviceManager::reserveStaging(size_t bytes) {
  // (at least as much as lets uploadInputs stage everything: a ranking request of 16
  // samples took 160 us by copies of its own for each of its 53 inputs)
  bytes = std::min(kStagingMost, std::max(kStagingLeast, (bytes + 4095) & ~(size_t)4095));
  int rc = MI355X_OK;
  if (!outputs_) rc = mi355x_host_alloc((void **)&outputs_, kOutputsMost);
  if (rc != MI355X_OK || bytes <= stagingBytes_) return rc;
  // (what is there stays until there is more, and does where there is none to be had)
  uint8_t *more = nullptr;
  rc = mi355x_host_alloc((void **)&more, bytes);
  if (rc != MI355X_OK && stagingBytes_ == 0)
    rc = mi355x_host_alloc((void **)&more, bytes = kStagingLeast);
  if (rc != MI355X_OK) return stagingBytes_ == 0 ? rc : (int)MI355X_OK;
  rc = mi355x_stream_sync(stream_);
  if (rc != MI355X_OK) {
    mi355x_host_free(more);
    return rc;
  }
  mi355x_host_free(staging_);
  staging_ = more;
  stagingBytes_ = bytes;
  return rc;
}

Error MI355XDeviceManager::makeResident(const Module *module, const std::string &name,
                                        MI355XFunction *fn) {
  const RuntimeBundle &rb = fn->getRuntimeBundle();
  // A function that writes a placeholder on the device and one that derives bag
  // positions from the host's copy of the same placeholder cannot share a module.
  for (const auto &f : functions_) {
    if (f.second.module != module) continue;
    for (const auto &w : fn->writtenPlaceholders)
      if (derivesFrom(*f.second.fn, w))
        return MI355X_MAKE_ERR(ErrorCode::DEVICE_FEATURE_NOT_SUPPORTED,
                               "function %s writes placeholder %s, from which resident function "
                               "%s takes bag positions made on the host: compile that one with "
                               "deriveBagOffsets off",
                               name.c_str(), w.c_str(), f.first.c_str());
    for (const auto &w : f.second.fn->writtenPlaceholders)
      if (derivesFrom(*fn, w))
        return MI355X_MAKE_ERR(ErrorCode::DEVICE_FEATURE_NOT_SUPPORTED,
                               "function %s takes bag positions made on the host from placeholder "
                               "%s, which resident function %s writes: compile it with "
                               "deriveBagOffsets off",
                               name.c_str(), w.c_str(), f.first.c_str());
  }
  ModuleResident &mr = modules_[module];
  if (!mr.arena && mr.users == 0) {
    int rc = mi355x_arena_create(module->constantsSize(), module->mutableSize(), 0, &mr.arena);
    if (rc != MI355X_OK) {
      modules_.erase(module);
      return fromStatus(rc, "module arena");
    }
    mr.bytes = mi355x_arena_bytes(mr.arena);
    usedMemoryBytes_ += mr.bytes;
    // placeholders start as zeros: the first (untimed) pass over a new network
    // runs before any request has filled them
    if (module->mutableSize()) {
      void *mp = nullptr;
      mi355x_arena_ptr(mr.arena, MI355X_REGION_MUTABLE, 0, &mp);
      mi355x_fill_u8(mp, 0, module->mutableSize(), stream_);
    }
    if (module->constantsSize()) {
      rc = mi355x_arena_upload(mr.arena, MI355X_REGION_CONSTANTS, 0,
                               module->constantsImage().data(), module->constantsSize(), stream_);
      if (rc == MI355X_OK) rc = mi355x_stream_sync(stream_);
      if (rc != MI355X_OK) {
        mi355x_arena_destroy(mr.arena);
        usedMemoryBytes_ -= mr.bytes;
        modules_.erase(module);
        return fromStatus(rc, "constants upload");
      }
    }
  }
  mr.users++;
  FunctionResident fr;
  fr.fn = fn;
  fr.module = module;
  auto failWith = [&](Error e) {
    release(fr);
    return e;
  };
  // (a quantized copy follows what requests upload: beside a function that writes the
  // input on the device its readers stay with the floats)
  bool quantizes = pool_->helpers() >= kQuantizeHelpers && !fn->quantizedInputs.empty() &&
                   !quantizesWhatIsWritten(*fn, *fn);
  for (const auto &f : functions_)
    if (f.second.module == module && quantizesWhatIsWritten(*fn, *f.second.fn)) quantizes = false;
  const size_t generated = rb.generatedConstantsMemSize + (quantizes ? quantizedBytes(*fn) : 0);
  int rc = mi355x_arena_create(generated, 0, rb.activationsMemSize, &fr.arena);
  if (rc != MI355X_OK) return failWith(fromStatus(rc, "function arena"));
  fr.bytes = mi355x_arena_bytes(fr.arena);
  usedMemoryBytes_ += fr.bytes;
  if (rb.activationsMemSize) {
    void *ap = nullptr;
    mi355x_arena_ptr(fr.arena, MI355X_REGION_ACTIVATIONS, 0, &ap);
    mi355x_fill_u8(ap, 0, rb.activationsMemSize, stream_);
  }
  void *p = nullptr;
  mi355x_arena_ptr(mr.arena, MI355X_REGION_CONSTANTS, 0, &p);
  fr.bindings.constants = (uint8_t *)p;
  mi355x_arena_ptr(mr.arena, MI355X_REGION_MUTABLE, 0, &p);
  fr.bindings.mutableMem = (uint8_t *)p;
  mi355x_arena_ptr(fr.arena, MI355X_REGION_CONSTANTS, 0, &p);
  fr.bindings.generated = (uint8_t *)p;
  mi355x_arena_ptr(fr.arena, MI355X_REGION_ACTIVATIONS, 0, &p);
  fr.bindings.activations = (uint8_t *)p;
  fr.bindings.stream = stream_;
  fr.bindings.opts.slws_math = config_.slwsMath;
  if (!fn->generated.empty()) {
    rc = mi355x_arena_upload(fr.arena, MI355X_REGION_CONSTANTS, 0, fn->generated.data(),
                             fn->generated.size(), stream_);
    if (rc != MI355X_OK) return failWith(fromStatus(rc, "generated constants upload"));
  }
  // float inputs that arrive quantized: from what their slots hold right now
  if (quantizes) {
    fr.bindings.quantized = fr.bindings.generated + alignUp(rb.generatedConstantsMemSize, 256);
    for (const auto &q : fn->quantizedInputs) {
      fr.quantized.push_back({(int8_t *)fr.bindings.quantized + q.at, q.elements, q.scale, q.offset});
      rc = quantizeSlot({fr.quantized.back()},
                        fr.bindings.mutableMem + rb.symbolTable.at(q.placeholder).offset,
                        q.elements * sizeof(float));
      if (rc != MI355X_OK) return failWith(fromStatus(rc, "quantized input"));
    }
  }
  // bag positions of lookups that take them with the lengths: from what the
  // lengths placeholders hold right now (zeros on a new module)
  for (const auto &d : fn->derivedBagOffsets) {
    auto st = rb.symbolTable.find(d.lengths);
    if (st == rb.symbolTable.end()) continue;
    rc = lengthsInSlot({{(int32_t *)d.ptr(fr.bindings), d.segments}},
                       fr.bindings.mutableMem + st->second.offset, st->second.size,
                       st->second.size);
    if (rc != MI355X_OK) return failWith(fromStatus(rc, "bag offsets"));
  }
  // pinned memory for a request that binds every input (256 bytes more per piece)
  size_t inputs = 0;
  for (const auto &kv : rb.symbolTable)
    if (kv.second.symbolCategory == SymbolCategory::Placeholder && kv.second.input)
      inputs += kv.second.size + kv.second.size / kStagePiece * 256 + 512;
  if (quantizes) inputs += fn->quantizedBytes + kStagePiece;
  rc = reserveStaging(inputs);
  if (rc != MI355X_OK) return failWith(fromStatus(rc, "pinned memory"));
  for (const auto &l : fn->setup) {
    rc = l.run(fr.bindings);
    if (rc != MI355X_OK) return failWith(fromStatus(rc, l.kernel.c_str()));
  }
  rc = mi355x_stream_sync(stream_);
  if (rc != MI355X_OK) return failWith(fromStatus(rc, "set-up launches"));
  if (config_.useLaunchGraphs) {
    // one eager pass first: entry points that allocate on first use must have
    // run before they are recorded
    {
      std::shared_lock<std::shared_mutex> tiles(fn->launchMutex());
      for (const auto &l : fn->launches) {
        rc = l.launch(fr.bindings);
        if (rc != MI355X_OK) return failWith(fromStatus(rc, l.kernel.c_str()));
      }
    }
    rc = mi355x_stream_sync(stream_);
    if (rc != MI355X_OK) return failWith(fromStatus(rc, "first pass"));
    if (config_.autotuneTiles) {
      Error te = tuneTiles(fn, fr.bindings);
      if (te) return failWith(std::move(te));
    }
    const int all = (int)sideStreams_.size() + 1;
    Error e = captureWithBranches(fr, all);
    if (e) return failWith(std::move(e));
    if (config_.autotuneBranches && all > 1) {
      fr.branchCandidates = {all, 1};
      if (all > 2) fr.branchCandidates.push_back(2);
      fr.branchCandidates.push_back(0);
      fr.branchesTuned = false;
    }
  }
  for (auto &f : functions_) {
    FunctionResident &reader = f.second;
    if (reader.module != module || !reader.bindings.quantized ||
        !quantizesWhatIsWritten(*reader.fn, *fn))
      continue;
    // its floats lie in their slots: it reads those from here on
    reader.bindings.quantized = nullptr;
    reader.quantized.clear();
    if (config_.useLaunchGraphs) {
      Error e = captureWithBranches(reader, reader.branches);
      if (e) {
        bindSlots(module);
        return failWith(std::move(e));
      }
    }
  }
  functions_.emplace(name, fr);
  bindSlots(module);
  return Error::success();
}

Error MI355XDeviceManager::captureWithBranches(FunctionResident &fr, int branches) {
  fr.branches = branches;
  if (branches == 0) {
    fr.fn->dropGraph(fr.bindings);
    return Error::success();
  }
  std::vector<void *> side(sideStreams_.begin(),
                           sideStreams_.begin() + std::min<size_t>(sideStreams_.size(),
                                                                   (size_t)std::max(0, branches - 1)));
  return fr.fn->captureGraph(fr.bindings, side);
}

// Runs one request. While the recordings of a function and its launches one by one are
// still being compared it also re-records and times as the phase says; every request
// computes the same results whichever serves it. A candidate is timed from the end of the
// request's pulls, as the request meets it: what the host does meanwhile counts where the
// device waits for it.
Error MI355XDeviceManager::executeTuned(FunctionResident &fr, ExecutionContext *ctx) {
  if (fr.branchesTuned) return fr.fn->execute(ctx);
  constexpr int kPerCandidate = 3;       // one warm-up and two timed requests
  const size_t cand = (size_t)(fr.branchPhase / kPerCandidate);
  const bool timed = fr.branchPhase % kPerCandidate != 0;
  Error err;
  if (!timed) {
    // candidate 0 is the recording made at load time
    if (cand > 0) err = captureWithBranches(fr, fr.branchCandidates[cand]);
    if (!err) err = fr.fn->execute(ctx);
  } else {
    void *e0 = nullptr, *e1 = nullptr;
    float ms = 0.0f;
    int rc = mi355x_event_create(&e0);
    if (rc == MI355X_OK) rc = mi355x_event_create(&e1);
    if (rc == MI355X_OK) rc = mi355x_event_record(e0, stream_);
    if (rc == MI355X_OK) {
      err = fr.fn->execute(ctx);
      if (!err) {
        rc = mi355x_event_record(e1, stream_);
        if (rc == MI355X_OK) rc = mi355x_event_sync(e1);
        if (rc == MI355X_OK) rc = mi355x_event_elapsed_ms(e0, e1, &ms);
      }
    }
    if (e0) mi355x_event_destroy(e0);
    if (e1) mi355x_event_destroy(e1);
    if (!err && rc != MI355X_OK) err = fromStatus(rc, "branch timing");
    if (!err) {
      if (fr.branchMs.size() <= cand) fr.branchMs.push_back(ms);
      else fr.branchMs[cand] = std::min(fr.branchMs[cand], ms);
    }
  }
  if (err) {
    // fall back to the recording with all branches and stop comparing
    fr.branchesTuned = true;
    Error again = captureWithBranches(fr, fr.branchCandidates[0]);
    (void)again;
    return err;
  }
  if (++fr.branchPhase == kPerCandidate * (int)fr.branchCandidates.size()) {
    size_t best = 0;
    for (size_t i = 1; i < fr.branchMs.size(); i++)
      if (fr.branchMs[i] < fr.branchMs[best] * (fr.branchCandidates[i] == 0 ? kDirectShare : 1.0f)) best = i;
    fr.branchesTuned = true;
    if (best + 1 != fr.branchCandidates.size())
      return captureWithBranches(fr, fr.branchCandidates[best]);
  }
  return Error::success();
}

// For every matrix-core launch: run each tile a few times on the resident data
// and keep the fastest (results do not depend on the tile).
Error MI355XDeviceManager::tuneTiles(MI355XFunction *fn, const DeviceBindings &b) {
  void *e0 = nullptr, *e1 = nullptr;
  int rc = mi355x_event_create(&e0);
  if (rc == MI355X_OK) rc = mi355x_event_create(&e1);
  Error err;
  // A launch of a few microseconds cannot be told from its neighbour by four
  // runs between two events: every candidate gets two series of kRuns launches
  // and its faster series counts. Three passes over the whole function first
  // bring the clocks up, so the first candidates are not timed on an idle part.
  constexpr int kRuns = 16, kSeries = 2;
  // (a copy: another device manager may be running the function)
  std::vector<KernelLaunch> launches;
  {
    std::shared_lock<std::shared_mutex> tiles(fn->launchMutex());
    launches = fn->launches;
  }
  for (int pass = 0; pass < 3 && rc == MI355X_OK; pass++)
    for (const auto &l : launches)
      if (rc == MI355X_OK) rc = l.launch(b);
  // seconds of kRuns launches of launch l with tile t (the faster of kSeries
  // series); negative when the tile cannot serve the launch
  auto timeTile = [&](KernelLaunch &l, int t) -> float {
    l.tile = t;
    if (l.launch(b) != MI355X_OK) return -1.0f;   // warm-up, also rejects tiles the shape cannot use
    float ms = 0.0f;
    for (int s = 0; s < kSeries && rc == MI355X_OK; s++) {
      rc = mi355x_event_record(e0, stream_);
      for (int i = 0; i < kRuns && rc == MI355X_OK; i++) rc = l.launch(b);
      if (rc == MI355X_OK) rc = mi355x_event_record(e1, stream_);
      if (rc == MI355X_OK) rc = mi355x_event_sync(e1);
      float one = 0.0f;
      if (rc == MI355X_OK) rc = mi355x_event_elapsed_ms(e0, e1, &one);
      if (s == 0 || one < ms) ms = one;
    }
    return ms;
  };
  for (size_t i = 0; i < launches.size(); i++) {
    KernelLaunch &l = launches[i];
    if (!l.tunable || rc != MI355X_OK) continue;
    float best = 0.0f;
    int bestTile = -1;
    for (int t = -1; t < kNumTiles && rc == MI355X_OK; t++) {
      const float ms = timeTile(l, t);
      if (ms < 0.0f) continue;
      if (rc == MI355X_OK && (t == -1 || ms < best)) {
        best = ms;
        bestTile = t;
      }
    }
    // A dozen candidates a few per cent apart: the fastest of one pass is often
    // a lucky measurement (several tile numbers run the very kernel the shape
    // rule picks). The winner has to beat the library's own choice again, by
    // two per cent, in a second pass, or that choice stays.
    if (bestTile != -1 && rc == MI355X_OK) {
      const float again = timeTile(l, bestTile), base = timeTile(l, -1);
      if (!(again >= 0.0f && base >= 0.0f && again < 0.98f * base)) bestTile = -1;
    }
    l.tile = bestTile;
    std::lock_guard<std::shared_mutex> tiles(fn->launchMutex());
    fn->launches[i].tile = bestTile;
  }
  if (rc != MI355X_OK) err = fromStatus(rc, "tile tuning");
  if (e0) mi355x_event_destroy(e0);
  if (e1) mi355x_event_destroy(e1);
  mi355x_stream_sync(stream_);
  return err;
}

void MI355XDeviceManager::addNetworkImpl(const Module *module, FunctionMapTy functions,
                                         ReadyCBTy readyCB) {
  uint64_t need = 0;
  for (const auto &f : functions) {
    if (functions_.count(f.first)) {
      readyCB(module, MI355X_MAKE_ERR(ErrorCode::RUNTIME_ERROR,
                                      "Failed to add network: already have a function called %s",
                                      f.first.c_str()));
      return;
    }
    if (!f.second || f.second->getCompileBackendName() != "MI355X") {
      readyCB(module, MI355X_MAKE_ERR(ErrorCode::RUNTIME_ERROR,
                                      "Failed to add network: function %s is not an MI355XFunction",
                                      f.first.c_str()));
      return;
    }
    const RuntimeBundle &rb = f.second->getRuntimeBundle();
    need += rb.generatedConstantsMemSize + rb.activationsMemSize;
    if (pool_->helpers() >= kQuantizeHelpers) need += quantizedBytes(*f.second);
  }
  if (!modules_.count(module)) need += module->constantsSize() + module->mutableSize();
  if (usedMemoryBytes_ + need > maxMemoryBytes_) {
    readyCB(module, MI355X_MAKE_ERR(ErrorCode::RUNTIME_OUT_OF_DEVICE_MEMORY,
                                    "Failed to add network: not enough memory (%llu needed, "
                                    "%llu available)",
                                    (unsigned long long)need,
                                    (unsigned long long)(maxMemoryBytes_ - usedMemoryBytes_)));
    return;
  }
  std::vector<std::string> added;
  for (const auto &f : functions) {
    Error e = makeResident(module, f.first, f.second);
    if (e) {
      for (const auto &n : added) {
        release(functions_[n]);
        functions_.erase(n);
      }
      bindSlots(module);
      readyCB(module, std::move(e));
      return;
    }
    added.push_back(f.first);
  }
  readyCB(module, Error::success());
}

void MI355XDeviceManager::evictNetworkImpl(std::string functionName, EvictFunctionCBTy evictCB) {
  auto it = functions_.find(functionName);
  if (it == functions_.end()) {
    evictCB(functionName, MI355X_MAKE_ERR(ErrorCode::RUNTIME_NET_NOT_FOUND,
                                          "Could not find function with name %s to evict",
                                          functionName.c_str()));
    return;
  }
  mi355x_stream_sync(stream_);
  const Module *module = it->second.module;
  release(it->second);
  functions_.erase(it);
  bindSlots(module);
  evictCB(functionName, Error::success());
}

// The request's inputs into their slots. Everything but large pinned tensors goes
// through pinned memory: copied there piece by piece by the pool (indices as 32
// bits where they fit: half the bytes over PCIe) and pulled by compute units as the
// pieces get ready. Small tensors first, so that their launch is not held up.
// What no launch waits for is left in `late`.
int MI355XDeviceManager::uploadInputs(std::vector<std::pair<Slot *, BoundArray>> &bound,
                                      std::vector<std::pair<Slot *, BoundArray>> &late) {
  std::vector<StagePiece> pieces;
  size_t used = 0;
  int rc = MI355X_OK;
  auto drain = [&] {
    if (pieces.empty()) return;
    std::vector<mi355x_copy_segment> segs;
    rc = pool_->run(pieces, staging_, [&](size_t first, size_t last) {
      segs.clear();
      for (size_t i = first; i < last; i++) segs.push_back(pieces[i].seg);
      return mi355x_copy_segments(segs.data(), segs.size(), nullptr, 0, nullptr, stream_);
    });
    pieces.clear();
    stagingUsed_ = used;
    used = 0;
  };
  stagingUsed_ = 0;
  auto add = [&](const uint8_t *src, size_t bytes, size_t staged,
                 const mi355x_copy_segment &seg) -> StagePiece & {
    const size_t room = (staged + 255) & ~(size_t)255;
    if (used + room > stagingBytes_) {
      // the device has to be done with what it pulls before it is overwritten
      drain();
      if (rc == MI355X_OK) rc = mi355x_stream_sync(stream_);
    }
    StagePiece p;
    p.src = src;
    p.bytes = bytes;
    p.at = used;
    p.seg = seg;
    pieces.push_back(p);
    used += room;
    return pieces.back();
  };
  std::stable_sort(bound.begin(), bound.end(), [](const auto &x, const auto &y) {
    return (x.second.bytes >= kStagePiece) < (y.second.bytes >= kStagePiece);
  });
  for (const auto &b : bound) {
    const Slot &s = *b.first;
    if (!s.input || rc != MI355X_OK) continue;
    const uint8_t *src = (const uint8_t *)b.second.data;
    const size_t bytes = b.second.bytes;
    if (!s.derived.empty()) {
      if (bytes > stagingBytes_ / 2 || bytes % sizeof(int32_t) != 0) {
        rc = mi355x_memcpy_h2d(s.device, src, bytes, stream_);
        if (rc == MI355X_OK) rc = lengthsInSlot(s.derived, s.device, s.bytes, bytes);
        continue;
      }
      // whole, with the positions that follow from it
      for (size_t k = 0; k < s.derived.size(); k++)
        add(src, bytes, bytes,
            {k == 0 ? s.device : nullptr, nullptr, 0, s.derived[k].positions,
             (uint32_t)s.derived[k].bags, MI355X_SEGMENT_LENGTHS})
            .form = StagePiece::Lengths;
      continue;
    }
    if (!s.quantized.empty() && bytes % sizeof(float) == 0) {
      for (const auto &q : s.quantized)
        for (size_t at = 0; at < bytes && rc == MI355X_OK; at += kStagePiece) {
          const size_t n = std::min(kStagePiece, bytes - at);
          StagePiece &p = add(src + at, n, n / 4,
                              {q.values + at / 4, nullptr, 0, nullptr, 0, MI355X_SEGMENT_COPY});
          p.form = StagePiece::Quantized;
          p.scale = q.scale;
          p.offset = (float)q.offset;
        }
      if (!s.floatRead) {
        late.push_back(b);
        continue;
      }
    }
    bool direct = false;
    if (!s.indices64 && bytes >= kDirectCopy) {
      int pinned = 0;
      direct = pool_->helpers() == 0 ||
               (mi355x_host_is_pinned(src, &pinned) == MI355X_OK && pinned);
    }
    if (direct) {
      rc = mi355x_memcpy_h2d(s.device, src, bytes, stream_);
      continue;
    }
    for (size_t at = 0; at < bytes && rc == MI355X_OK; at += kStagePiece) {
      const size_t n = std::min(kStagePiece, bytes - at);
      StagePiece &p = add(src + at, n, n,
                          {s.device + at, nullptr, 0, nullptr, 0, MI355X_SEGMENT_COPY});
      if (s.indices64 && bytes % 8 == 0) p.form = StagePiece::Indices64;
    }
  }
  if (rc == MI355X_OK) drain();
  // a float tensor cut off inside a value: quantized from its slot after all
  for (const auto &b : bound)
    if (b.first->input && !b.first->quantized.empty() && b.second.bytes % sizeof(float) != 0 &&
        rc == MI355X_OK)
      rc = quantizeSlot(b.first->quantized, b.first->device, b.second.bytes);
  for (const auto &b : bound)
    if (b.first->input && rc == MI355X_OK) rc = refreshOverlapped(*b.first);
  return rc;
}

// The float values of inputs that the launches take quantized, while those run: a
// function loaded later, a shorter tensor or a writer of the placeholder finds them in
// the slot. By the DMA engines, which leave the compute units alone.
int MI355XDeviceManager::uploadLate(const std::vector<std::pair<Slot *, BoundArray>> &late) {
  int rc = MI355X_OK;
  size_t used = stagingUsed_;
  for (const auto &b : late) {
    uint8_t *dst = b.first->device;
    const uint8_t *src = (const uint8_t *)b.second.data;
    const size_t bytes = b.second.bytes;
    int pinned = 0;
    if (bytes >= kDirectCopy && (mi355x_host_is_pinned(src, &pinned) == MI355X_OK && pinned)) {
      if (rc == MI355X_OK) rc = mi355x_memcpy_h2d(dst, src, bytes, lateStream_);
      continue;
    }
    std::vector<StagePiece> pieces;
    for (size_t at = 0; at < bytes && rc == MI355X_OK;) {
      if (used + kStagePiece > stagingBytes_) {
        // from the front again, once nothing there is waited for any more
        rc = mi355x_stream_sync(lateStream_);
        if (rc == MI355X_OK && stagingUsed_ + kStagePiece > stagingBytes_) {
          rc = mi355x_stream_sync(stream_);
          stagingUsed_ = 0;
        }
        used = stagingUsed_;
      }
      pieces.clear();
      const size_t from = at;
      for (; at < bytes && used + kStagePiece <= stagingBytes_; at += kStagePiece, used += kStagePiece) {
        StagePiece p;
        p.src = src + at;
        p.bytes = std::min(kStagePiece, bytes - at);
        p.at = used;
        pieces.push_back(p);
      }
      // pieces lie one behind the other on both sides: a copy for every few of them
      size_t sent = 0;
      if (rc == MI355X_OK)
        rc = pool_->run(pieces, staging_, [&](size_t, size_t last) {
          const size_t end = last == pieces.size() ? std::min(at, bytes) - from : last * kStagePiece;
          if (last < pieces.size() && end - sent < kLateCopy) return (int)MI355X_OK;
          const int e = mi355x_memcpy_h2d(dst + from + sent, staging_ + pieces[0].at + sent, end - sent,
                                          lateStream_);
          sent = end;
          return e;
        });
    }
  }
  return rc;
}

// The request's outputs, and the end of the request: returns when everything
// queued for it has finished and the callers' arrays hold their values.
int MI355XDeviceManager::downloadOutputs(const std::vector<std::pair<Slot *, BoundArray>> &bound) {
  std::vector<mi355x_copy_segment> segs;
  struct Staged {
    void *to;
    size_t at, bytes;
  };
  std::vector<Staged> staged;
  size_t used = 0;
  bool direct = false;
  int rc = MI355X_OK;
  for (const auto &b : bound) {
    if (!b.first->output || rc != MI355X_OK) continue;
    const size_t bytes = std::min(b.second.bytes, b.first->bytes);
    if (bytes == 0) continue;
    if (used + bytes > kOutputsMost) {
      rc = mi355x_memcpy_d2h(b.second.data, b.first->device, bytes, stream_);
      direct = true;
      continue;
    }
    segs.push_back({outputs_ + used, b.first->device, bytes, nullptr, 0, MI355X_SEGMENT_COPY});
    staged.push_back({b.second.data, used, bytes});
    used += (bytes + 255) & ~(size_t)255;
  }
  if (rc == MI355X_OK && !segs.empty() && !direct) {
    rc = mi355x_copy_segments(segs.data(), segs.size(), done_, ++doneValue_, arrived_, stream_);
    if (rc == MI355X_OK) rc = waitForDevice();
  } else {
    if (rc == MI355X_OK && !segs.empty())
      rc = mi355x_copy_segments(segs.data(), segs.size(), nullptr, 0, nullptr, stream_);
    const int sync = mi355x_stream_sync(stream_);
    if (rc == MI355X_OK) rc = sync;
  }
  if (rc == MI355X_OK)
    for (const auto &o : staged) std::memcpy(o.to, outputs_ + o.at, o.bytes);
  return rc;
}

// Waits for the word that the last launch of a request sets; a look at the stream
// now and then ends the wait should the device have failed.
int MI355XDeviceManager::waitForDevice() {
  for (;;) {
    for (int i = 0; i < 2000; i++) {
      if (__atomic_load_n(done_, __ATOMIC_ACQUIRE) == doneValue_) return MI355X_OK;
      __builtin_ia32_pause();
    }
    int idle = 0;
    const int rc = mi355x_stream_query(stream_, &idle);
    if (rc != MI355X_OK || idle) return rc;
  }
}

Error MI355XDeviceManager::runRequest(const std::string &functionName, const BoundArray *arrays,
                                      size_t n) {
  auto it = functions_.find(functionName);
  if (it == functions_.end())
    return MI355X_MAKE_ERR(ErrorCode::RUNTIME_NET_NOT_FOUND, "Function %s not found",
                           functionName.c_str());
  FunctionResident &fr = it->second;
  Error err;
  // a tensor smaller than its slot fills the slot's front, like the reference's
  // partial tensors; of two bindings of one name the later counts
  std::vector<std::pair<Slot *, BoundArray>> bound;
  bound.reserve(n);
  requests_++;
  for (size_t i = 0; i < n && !err; i++) {
    auto st = fr.slots.find(arrays[i].name);
    if (st == fr.slots.end()) continue;
    Slot &s = st->second;
    if (s.input && arrays[i].bytes > s.bytes)
      err = MI355X_MAKE_ERR(ErrorCode::RUNTIME_ERROR, "tensor bound to %s has %zu bytes, slot %zu",
                            arrays[i].name, arrays[i].bytes, s.bytes);
    if (s.request == requests_) {
      bound[s.at].second = arrays[i];
      continue;
    }
    s.request = requests_;
    s.at = bound.size();
    bound.push_back({&s, arrays[i]});
  }
  if (err) return err;
  std::vector<std::pair<Slot *, BoundArray>> late;
  int rc = uploadInputs(bound, late);
  if (rc != MI355X_OK) err = fromStatus(rc, "input copy");
  if (!err) {
    ExecutionContext ctx;
    ctx.setDeviceBindings(std::unique_ptr<DeviceBindings>(new DeviceBindings(fr.bindings)));
    err = executeTuned(fr, &ctx);
    rc = uploadLate(late);
    if (rc != MI355X_OK && !err) err = fromStatus(rc, "input copy");
  }
  if (!err) {
    rc = downloadOutputs(bound);
    if (rc != MI355X_OK) err = fromStatus(rc, "output copy");
  }
  // nothing of the request is left running
  if (!late.empty()) {
    rc = mi355x_stream_sync(lateStream_);
    if (rc != MI355X_OK && !err) err = fromStatus(rc, "input copy");
  }
  if (err) mi355x_stream_sync(stream_);
  return err;
}

} // namespace glow_mi355x
