// Work of the host for the time a call waits for the device: what an operator's caller has to do anyway and the device need not
// wait for.
#ifndef TN_HOST_WORK_H_
#define TN_HOST_WORK_H_

extern "C" {

// The calling thread's next operator calls fn(arg) once, with its launches queued, before it waits for what they report; not at
// all if it does not get there.  fn: nullptr takes it back.  fn must not throw, nor call this library.
__attribute__((visibility("default"))) void tn_while_waiting(void (*fn)(void*), void* arg);
}

#endif  // TN_HOST_WORK_H_
