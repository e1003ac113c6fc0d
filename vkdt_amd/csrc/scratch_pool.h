// scratch_pool.h -- a bounded pool of device blocks and pinned staging
// buffers for the codec entry points, over a memory M given as static
// functions (the HIP runtime in exec.hip, counters in the test):
//   int device(int *)            the calling thread's device
//   int dev_alloc(void **, size_t), void dev_free(void *)
//   int pin_alloc(void **, size_t), void pin_free(void *)
//   bool oom(int)                whether that error is a lack of memory
//   void forget()                clears the error that the thread last had
// Errors are M's, 0 is success.  Nothing here throws: the callers are C entry
// points, and the idle blocks lie in arrays of fixed size.
#pragma once
#include <stddef.h>
#include <stdint.h>
#include <mutex>

struct scratch_t
{
  uint8_t *dev;      // device memory of at least the bytes asked for
  uint8_t *pin;      // SCRATCH_PINNED bytes of pinned host memory, where asked for
  size_t   size;
  int      device;
};

// The pool keeps at most SCRATCH_KEEP bytes of idle device memory, so that the
// two blocks of a 61 MP export in 4:4:4 (367 MB of coefficients, up to 270 MB
// of stream) stay from one to the next: of a card's 288 GB, given back when an
// allocation fails
#define SCRATCH_KEEP ((size_t)1 << 30)
#define SCRATCH_PINNED ((size_t)64 << 10)
#define SCRATCH_SLOTS 64

template<typename M>
class scratch_pool
{
public:
  // a block of at least `bytes`, with a pinned buffer where asked for.  A
  // failure leaves s empty: putting it back is no harm
  int get(scratch_t &s, size_t bytes, bool pinned)
  {
    s = scratch_t{};
    scratch_t b = {};
    if(int e = M::device(&b.device)) return e;
    // whole megabytes, so that images of about one size share blocks
    b.size = (bytes + ((size_t)1 << 20)) & ~(((size_t)1 << 20) - 1);
    {
      std::lock_guard<std::mutex> lk(mx);
      int best = -1;
      for(int k = 0; k < n; k++)
        if(idle[k].device == b.device && idle[k].size >= b.size && idle[k].size <= 2 * b.size &&
           (best < 0 || idle[k].size < idle[best].size))
          best = k;
      if(best >= 0) b = take(best);
    }
    if(!b.dev)
      if(int e = alloc(M::dev_alloc, (void **)&b.dev, b.size)) return e;
    if(pinned && !b.pin)
      if(int e = alloc(M::pin_alloc, (void **)&b.pin, SCRATCH_PINNED))
      {
        M::dev_free(b.dev);
        return e;
      }
    s = b;
    return 0;
  }

  // ok: the stream has drained and the next user may take the block at once;
  // else it is freed, which waits for it
  void put(scratch_t &s, bool ok)
  {
    if(!s.dev) return;
    scratch_t out[SCRATCH_SLOTS + 1];
    int no = 0;
    if(!ok || s.size > SCRATCH_KEEP) out[no++] = s;
    else
    {
      std::lock_guard<std::mutex> lk(mx);
      while(n && (n == SCRATCH_SLOTS || kept + s.size > SCRATCH_KEEP)) out[no++] = take(0);   // the oldest
      idle[n++] = s;
      kept += s.size;
    }
    for(int k = 0; k < no; k++) free_block(out[k]);
    s = scratch_t{};
  }

  // gives the idle blocks back; false if there were none
  bool trim()
  {
    scratch_t out[SCRATCH_SLOTS];
    int no = 0;
    {
      std::lock_guard<std::mutex> lk(mx);
      while(n) out[no++] = take(n - 1);
    }
    for(int k = 0; k < no; k++) free_block(out[k]);
    return no > 0;
  }

  // an allocation, tried again without the idle blocks where memory lacks.  Its
  // error is forgotten, whether the second try succeeds or the caller is told:
  // the runtime keeps it through later successful calls, and the check of the
  // next launch would read it
  template<typename F>
  int alloc(F f, void **p, size_t bytes)
  {
    int e = f(p, bytes);
    if(e) M::forget();
    if(e && M::oom(e) && trim())
    {
      e = f(p, bytes);
      if(e) M::forget();
    }
    return e;
  }

private:
  std::mutex mx;
  scratch_t idle[SCRATCH_SLOTS];   // oldest first
  int n = 0;
  size_t kept = 0;

  scratch_t take(int k)
  {
    const scratch_t b = idle[k];
    n--;
    for(; k < n; k++) idle[k] = idle[k + 1];
    kept -= b.size;
    return b;
  }

  static void free_block(const scratch_t &s)
  {
    M::dev_free(s.dev);
    if(s.pin) M::pin_free(s.pin);
  }
};
