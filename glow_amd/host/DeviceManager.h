// MI355XDeviceManager: owns one GPU's resident networks and runs them.
// Mirrors glow::runtime::DeviceManager / QueueBackedDeviceManager (reference
// include/glow/Backends/DeviceManager.h:47-241,
// include/glow/Backends/QueueBackedDeviceManager.h:30-127) and the behaviour of
// CPUDeviceManager (lib/Backends/CPU/CPUDeviceManager.cpp:65-177): work runs one
// piece at a time, on a worker thread or on the thread of a caller who waits for a
// request anyway; results come back through callbacks, errors are values. Whoever runs
// a request is awake until it is over (it watches a word that the last launch sets),
// and helper threads stage the request's inputs beside it (Staging.h). One compiled
// function may be on several device managers at once.
#ifndef GLOW_MI355X_HOST_DEVICEMANAGER_H
#define GLOW_MI355X_HOST_DEVICEMANAGER_H

#include "Backend.h"
#include "Staging.h"

#include <atomic>
#include <condition_variable>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <thread>
#include <unordered_map>

struct mi355x_arena;

namespace glow_mi355x {

using RunIdentifierTy = uint64_t;
using FunctionMapTy = std::map<std::string, MI355XFunction *>;
using ReadyCBTy = std::function<void(const Module *, Error)>;
using EvictFunctionCBTy = std::function<void(std::string, Error)>;
using ResultCBTy = std::function<void(RunIdentifierTy, Error, std::unique_ptr<ExecutionContext>)>;

struct DeviceConfig {
  int deviceID = 0;
  uint64_t deviceMemory = 0;  // 0 = what the device reports as free at init
  bool useLaunchGraphs = true; // record each function, replay per run
  int graphBranches = 4;       // independent launches recorded side by side (1 = a chain)
  bool autotuneTiles = true;   // time the tile candidates of each matrix-core launch at load
  // The first requests of a function replay it recorded with all branches, as
  // one chain and with two branches, then issue its launches one by one (a warm-up
  // and two timed requests each); the fastest serves the requests after them.
  // Waiting for another stream costs microseconds, so short side branches can lose
  // more than they overlap, and how long a launch runs depends on the request's data.
  // A graph of 14 launches takes the host 24 us to replay and the device another 10
  // before its first launch, the first of single launches 3 (a ranking request of 4096
  // samples 287 / 272 us); of 58 launches, an image network answering one image, the
  // two are level.
  bool autotuneBranches = true;
  // Arithmetic of this device manager's SparseLengths launches, passed with
  // every such call (mi355x_launch_opts::slws_math): MI355X_SLWS_MATH_*, or -1
  // for the library's default.
  int slwsMath = -1;
};

struct DeviceInfo {
  std::string name, arch;
  uint64_t totalMemory = 0;
  int computeUnits = 0;
};

// A caller's array bound to a placeholder for one request.
struct BoundArray {
  const char *name;
  void *data;
  size_t bytes;
};

class MI355XDeviceManager {
public:
  explicit MI355XDeviceManager(const DeviceConfig &config) : config_(config) {}
  ~MI355XDeviceManager();

  // Starts the worker thread and binds the device; RUNTIME_DEVICE_NOT_FOUND
  // when there is no such gfx950 device.
  Error init();
  // Drains the queue, frees every network, stops the worker.
  Error stop(bool block = true);

  // Asynchronous: the callback runs on the worker thread.
  void addNetwork(const Module *module, FunctionMapTy functions, ReadyCBTy readyCB);
  void evictNetwork(std::string functionName, EvictFunctionCBTy evictCB);
  RunIdentifierTy runFunction(std::string functionName, std::unique_ptr<ExecutionContext> ctx,
                              ResultCBTy resultCB);
  // runFunction for a caller that waits for the result anyway: runs on the calling
  // thread when the manager has nothing else to do (two hand-overs between threads
  // less, 15 us), behind what is queued otherwise.
  Error runFunctionBlocking(const char *functionName, const BoundArray *arrays, size_t n);

  // DeviceManager::transferStaticPlaceholderToDevice (reference
  // include/glow/Backends/DeviceManager.h:166-171): copies `tensor` into the
  // device slot of the module's placeholder `placeholderName`. Requests that
  // do not bind that placeholder afterwards run on the transferred value (a
  // static placeholder: uploaded once, read by many requests). The module must
  // have a function resident on this device; a tensor larger than the slot, an
  // unknown name or a value that is no placeholder is a RUNTIME_ERROR.
  void transferStaticPlaceholderToDevice(const Module *module, std::string placeholderName,
                                         Tensor *tensor, std::function<void(Error)> resultCB);

  // Benchmark aid without a counterpart in the reference: replays a resident
  // function `iterations` times on the data its placeholders already hold (no
  // host copies) and reports the average device time per replay, measured
  // with events on the manager's stream. Blocks until done.
  Expected<float> timeFunction(const std::string &functionName, int iterations);
  // How many branches the recording has that serves the function's requests now; 0: its
  // launches are issued one by one.
  Expected<int> recordedBranches(const std::string &functionName);

  uint64_t getMaximumMemory() const { return maxMemoryBytes_; }
  uint64_t getAvailableMemory() const { return maxMemoryBytes_ - usedMemoryBytes_; }
  bool isMemoryAvailable(uint64_t estimate) const {
    return maxMemoryBytes_ >= usedMemoryBytes_ + estimate;
  }
  DeviceInfo getDeviceInfo() const { return info_; }
  std::string getBackendName() const { return "MI355X"; }

private:
  struct ModuleResident {   // constants + placeholders of one module
    mi355x_arena *arena = nullptr;
    uint64_t bytes = 0;
    int users = 0;
  };
  // What a request may bind: a placeholder's place on the device, and the vectors of
  // bag positions derived from it (of any resident function of the module).
  struct DerivedPositions {
    int32_t *positions;
    size_t bags;
  };
  struct QuantizedCopy {   // a float placeholder as int8, where a launch reads it
    int8_t *values;
    size_t elements;
    float scale;
    int32_t offset;
  };
  struct Slot {
    uint8_t *device = nullptr;
    size_t bytes = 0;
    bool input = false, output = false, indices64 = false;
    std::vector<DerivedPositions> derived;
    std::vector<QuantizedCopy> quantized;
    // false: every reader that is loaded takes one of `quantized`, and a request's float
    // values may follow behind its launches (a function loaded later may read them)
    bool floatRead = true;
    // slots with copies or positions of their own that share memory with this one (a
    // view and what it views): made again from their slots when this one is filled
    std::vector<const Slot *> overlapped;
    uint64_t request = 0;  // the last request that bound it, and where in its list
    size_t at = 0;
  };
  struct FunctionResident {
    MI355XFunction *fn = nullptr;
    const Module *module = nullptr;
    mi355x_arena *arena = nullptr; // generated constants + activations
    uint64_t bytes = 0;
    DeviceBindings bindings;
    // branch tuning: requests 3c, 3c+1, 3c+2 go to candidate c (warm-up, timed, timed)
    std::vector<int> branchCandidates;
    std::vector<float> branchMs;
    int branchPhase = 0;
    bool branchesTuned = true;
    int branches = 1;             // of the present recording; 0: launched one by one
    std::unordered_map<std::string, Slot> slots;
    std::vector<QuantizedCopy> quantized; // of fn->quantizedInputs, in this arena
  };

  void addNetworkImpl(const Module *module, FunctionMapTy functions, ReadyCBTy readyCB);
  void evictNetworkImpl(std::string functionName, EvictFunctionCBTy evictCB);
  Error runRequest(const std::string &functionName, const BoundArray *arrays, size_t n);
  int uploadInputs(std::vector<std::pair<Slot *, BoundArray>> &bound,
                   std::vector<std::pair<Slot *, BoundArray>> &late);
  int uploadLate(const std::vector<std::pair<Slot *, BoundArray>> &late);
  int downloadOutputs(const std::vector<std::pair<Slot *, BoundArray>> &bound);
  int waitForDevice();
  void bindSlots(const Module *module);
  int reserveStaging(size_t bytes);
  Error makeResident(const Module *module, const std::string &name, MI355XFunction *fn);
  Error tuneTiles(MI355XFunction *fn, const DeviceBindings &b);
  Error captureWithBranches(FunctionResident &fr, int branches);
  Error executeTuned(FunctionResident &fr, ExecutionContext *ctx);
  void release(FunctionResident &fr);
  void enqueue(std::function<void()> work);
  int quantizeSlot(const std::vector<QuantizedCopy> &copies, const uint8_t *slot, size_t bytes);
  int refreshOverlapped(const Slot &s);
  int lengthsInSlot(const std::vector<DerivedPositions> &derived, uint8_t *slot, size_t slotBytes,
                    size_t bytes);
  void workerLoop();

  DeviceConfig config_;
  DeviceInfo info_;
  std::atomic<uint64_t> maxMemoryBytes_{0}, usedMemoryBytes_{0};
  std::atomic<RunIdentifierTy> nextRun_{1};
  std::map<std::string, FunctionResident> functions_;
  std::map<const Module *, ModuleResident> modules_;
  void *stream_ = nullptr;
  std::vector<void *> sideStreams_; // branches of captured graphs
  void *lateStream_ = nullptr;      // inputs that no launch of their request reads

  // Pinned memory that requests pass through: inputs (staged by pool_), the
  // outputs of one request, and the word the last launch of a request sets.
  std::unique_ptr<StagingPool> pool_;
  uint8_t *staging_ = nullptr;
  size_t stagingBytes_ = 0;
  size_t stagingUsed_ = 0; // of the last request's inputs, that it may still pull
  uint8_t *outputs_ = nullptr;
  uint32_t *done_ = nullptr;
  uint32_t doneValue_ = 0;
  uint32_t *arrived_ = nullptr; // device
  uint64_t requests_ = 0;

  std::thread worker_;
  std::mutex mu_;
  std::condition_variable cv_;
  std::deque<std::function<void()>> queue_;
  bool running_ = false, stopping_ = false;
  bool busy_ = false; // the worker, or a caller in its place, is at work
};

} // namespace glow_mi355x
#endif
