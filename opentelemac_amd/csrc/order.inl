// Ordering of a context's stream with one of the caller's, on the device.

namespace bhip {

// Makes `dev` the current device for as long as it lives.
class DeviceScope {
 public:
  hipError_t enter(int dev) {
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess || cur == dev) return e;
    e = hipSetDevice(dev);
    if (e == hipSuccess) back_ = cur;
    return e;
  }
  ~DeviceScope() {
    if (back_ >= 0) (void)hipSetDevice(back_);
  }

 private:
  int back_ = -1;
};

// One event serves all recordings on streams of the context's device (a wait
// keeps the recording it was given). An event records on streams of the device
// it was created on only, whatever the current one is, so streams of other
// devices take one of their own.
struct StreamOrder {
  std::mutex mu;
  hipEvent_t ev = nullptr;

  // `second` after what `first`, a stream of device first_dev, holds now
  hipError_t after(int ctx_dev, hipStream_t first, int first_dev, hipStream_t second) {
    if (first == second) return hipSuccess;
    if (first_dev != ctx_dev) {
      hipEvent_t one;
      {
        DeviceScope on;
        hipError_t e = on.enter(first_dev);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&one, hipEventDisableTiming);
        if (e != hipSuccess) return e;
      }
      hipError_t e = hipEventRecord(one, first);
      if (e == hipSuccess) e = hipStreamWaitEvent(second, one, 0);
      (void)hipEventDestroy(one);
      return e;
    }
    std::lock_guard<std::mutex> use(mu);
    if (!ev) {
      DeviceScope on;
      hipError_t e = on.enter(ctx_dev);
      if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
      if (e != hipSuccess) return e;
    }
    const hipError_t e = hipEventRecord(ev, first);
    return e == hipSuccess ? hipStreamWaitEvent(second, ev, 0) : e;
  }

  // the device of a caller's stream (the null stream is the current device's)
  static hipError_t device_of(hipStream_t s, int* dev) {
    return s ? hipStreamGetDevice(s, dev) : hipGetDevice(dev);
  }
};

}  // namespace bhip
