// Work of the host for the time a call waits for the device: what an operator's caller has to do anyway and the device need not
// wait for.
#ifndef TN_HOST_WORK_H_
#define TN_HOST_WORK_H_

extern "C" {

// The calling thread's next call that waits for the device -- a pull, of a batch or of the table, or a combine -- calls fn(arg)
// once, with its launches queued, before it waits for what they report.  Other calls (a push, a pull that does not wait, one
// that is refused) leave it for the next one.  fn: nullptr takes it back.
// fn runs under the lock of the call's table: other threads' calls on that table wait for it.  It must not throw, nor call
// this library, nor wait for a thread that may be in it.
__attribute__((visibility("default"))) void tn_while_waiting(void (*fn)(void*), void* arg);
}

#endif  // TN_HOST_WORK_H_
