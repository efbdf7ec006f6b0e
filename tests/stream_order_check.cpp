// StreamOrder over a model of HIP with two devices: events record on streams of
// the device they were created on only. Prints "ok" or what is wrong.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <mutex>

struct ihipStream_t {
  int dev;
  int after = -1;  // device of the stream that this one was last ordered after
};
struct ihipEvent_t {
  int dev;
  int recorded = -1;
};
static int current = 0, events = 0, ordered_null = -1;

extern "C" {
hipError_t hipGetDevice(int* d) {
  *d = current;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  current = d;
  return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) {
  *d = s ? s->dev : current;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new ihipEvent_t{current};
  ++events;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  --events;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  const int dev = s ? s->dev : current;
  if (e->dev != dev) return hipErrorInvalidHandle;
  e->recorded = dev;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  if (e->recorded < 0) return hipErrorInvalidValue;
  (s ? s->after : ordered_null) = e->recorded;
  return hipSuccess;
}
}

#include "order.inl"

int main() {
  for (int ctx_dev = 0; ctx_dev < 2; ++ctx_dev)
    for (int cur = 0; cur < 2; ++cur)
      for (int which = -1; which < 2; ++which)  // caller's stream: null, of device 0, of 1
        for (int turn = 0; turn < 2; ++turn) {  // which direction first makes the event
          bhip::StreamOrder o;
          ihipStream_t own{ctx_dev}, other{which};
          hipStream_t caller = which < 0 ? nullptr : &other;
          const int caller_dev = which < 0 ? cur : which;
          current = cur;
          for (int k = 0; k < 4; ++k) {
            own.after = other.after = ordered_null = -1;
            hipError_t e;
            int dev = -1;
            if ((k + turn) & 1) {
              e = bhip::StreamOrder::device_of(caller, &dev);
              if (e == hipSuccess) e = o.after(ctx_dev, caller, dev, &own);
              if (e == hipSuccess && own.after != caller_dev) e = hipErrorUnknown;
            } else {
              e = o.after(ctx_dev, &own, ctx_dev, caller);
              if (e == hipSuccess && (caller ? other.after : ordered_null) != ctx_dev)
                e = hipErrorUnknown;
            }
            if (e != hipSuccess || current != cur || events > 1) {
              printf("context on %d, current %d, stream of %d, call %d: error %d, current now %d, "
                     "%d events\n", ctx_dev, cur, which, k, (int)e, current, events);
              return 1;
            }
          }
          if (o.ev) (void)hipEventDestroy(o.ev);
          if (events) {
            printf("%d events left\n", events);
            return 1;
          }
        }
  printf("ok\n");
  return 0;
}
