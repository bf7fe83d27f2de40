// A stream's work recorded into a HIP graph, with a memory pool of its own (torch.classes.llmctl.StepCapture): training steps, which draw no random numbers.
// torch's CUDAGraph marks the default generator as captured for as long as it records, so a draw of another thread fails meanwhile, and keeps its seed in tensors that
// belong to the mode (inference or not) in which the first graph was recorded.
#include <ATen/hip/HIPContext.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGuard.h>
#include <hip/hip_runtime_api.h>
#include <torch/custom_class.h>
#include <torch/library.h>

#include <cstdint>

namespace llmctl {
namespace {

void check(hipError_t e, const char* what) {
  if (e == hipSuccess) return;
  (void)hipGetLastError();
  TORCH_CHECK(false, "llmctl: step capture: ", what, ": ", hipGetErrorString(e));
}

class StepCapture : public torch::CustomClassHolder {
 public:
  // pool: what torch.cuda.graph_pool_handle() gave; graphs that run one after the other may share one
  StepCapture(int64_t pool0, int64_t pool1) : pool_{(c10::CaptureId_t)pool0, (c10::CaptureId_t)pool1} {}
  ~StepCapture() override { release(); }

  // Record what reaches the current stream (none of the device's default one) and those that wait for it, from any thread; other threads go on working.
  void begin() {
    TORCH_CHECK(state_ == NEW, "llmctl: step capture: recorded once");
    device_ = c10::hip::current_device();
    const hipStream_t s = at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
    check(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal), "begin");
    stream_ = s;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    const hipError_t e = hipStreamGetCaptureInfo(s, &status, &id);
    if (e != hipSuccess) {
      hipGraph_t g = nullptr;
      if (hipStreamEndCapture(s, &g) == hipSuccess && g != nullptr) (void)hipGraphDestroy(g);
      check(e, "id");
    }
    c10::hip::HIPCachingAllocator::beginAllocateToPool(device_, pool_, [id](hipStream_t t) {
      hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
      unsigned long long of = 0;
      if (hipStreamGetCaptureInfo(t, &st, &of) == hipSuccess) return st == hipStreamCaptureStatusActive && of == id;
      (void)hipGetLastError();
      return false;
    });
    state_ = RECORDING;
  }

  void end() {
    TORCH_CHECK(state_ == RECORDING, "llmctl: step capture: not recording");
    state_ = ENDED;
    c10::hip::HIPCachingAllocator::endAllocateToPool(device_, pool_);
    check(hipStreamEndCapture(stream_, &graph_), "end");
    TORCH_CHECK(graph_ != nullptr, "llmctl: step capture: the recording was given up");
  }

  int64_t graph() const { return (int64_t)reinterpret_cast<uintptr_t>(graph_); }

  void instantiate() {
    TORCH_CHECK(graph_ != nullptr && exec_ == nullptr, "llmctl: step capture: nothing recorded");
    check(hipGraphInstantiate(&exec_, graph_, nullptr, nullptr, 0), "instantiate");
  }

  // on the current stream
  void replay() {
    TORCH_CHECK(exec_ != nullptr, "llmctl: step capture: nothing to replay");
    const c10::hip::HIPGuard guard(device_);
    check(hipGraphLaunch(exec_, at::hip::getCurrentHIPStreamMasqueradingAsCUDA(device_).stream()), "launch");
  }

  // Waits for the last replay: the pool's memory goes back to the allocator.
  void release() noexcept {
    if (state_ == NEW || state_ == RELEASED) return;
    int before = -1;
    (void)hipGetDevice(&before);
    (void)hipSetDevice(device_);
    try {
      if (state_ == RECORDING) {
        c10::hip::HIPCachingAllocator::endAllocateToPool(device_, pool_);
        (void)hipStreamEndCapture(stream_, &graph_);
      }
      if (exec_ != nullptr) {
        (void)hipDeviceSynchronize();
        (void)hipGraphExecDestroy(exec_);
      }
      if (graph_ != nullptr) (void)hipGraphDestroy(graph_);
      c10::hip::HIPCachingAllocator::releasePool(device_, pool_);
    } catch (...) {  // (called by a destructor)
    }
    (void)hipGetLastError();
    if (before >= 0) (void)hipSetDevice(before);
    exec_ = nullptr, graph_ = nullptr, state_ = RELEASED;
  }

 private:
  enum { NEW, RECORDING, ENDED, RELEASED } state_ = NEW;
  c10::MempoolId_t pool_;
  c10::DeviceIndex device_ = -1;
  hipStream_t stream_ = nullptr;
  hipGraph_t graph_ = nullptr;
  hipGraphExec_t exec_ = nullptr;
};

}  // namespace

TORCH_LIBRARY_FRAGMENT(llmctl, m) {
  m.class_<StepCapture>("StepCapture")
      .def(torch::init<int64_t, int64_t>())
      .def("begin", &StepCapture::begin)
      .def("end", &StepCapture::end)
      .def("graph", &StepCapture::graph)
      .def("instantiate", &StepCapture::instantiate)
      .def("replay", &StepCapture::replay)
      .def("release", [](const c10::intrusive_ptr<StepCapture>& c) { c->release(); });
}

}  // namespace llmctl
