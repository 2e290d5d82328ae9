// Which stream owns which K-split workspace of a context.
//
// Every stream has its own, so that a caller who moves one context between
// streams need not order their launches.  At most SLOTS streams hold one at a
// time; a stream past them goes without until one of theirs has been idle for
// IDLE requests of the whole table (streams come and go, torch hands out 32 a
// device).  A slot changes hands only after the device has been waited for: its
// old stream may have work in flight, or be gone.  A refused allocation is
// remembered and tried again after as many requests.
#pragma once
#include <cstdint>

namespace mk {

struct WsTable {
  static constexpr int SLOTS = 16;
  static constexpr uint64_t IDLE = 1024;
  struct Slot {
    const void* stream = nullptr;
    void* ptr = nullptr;
    uint64_t used = 0, tried = 0;
  };
  Slot slot[SLOTS];
  int n = 0;
  uint64_t clock = 0;

  // The workspace of `stream`, or null.  alloc() returns memory or null; wait()
  // waits for the device and tells whether that went well.
  template <class Alloc, class Wait>
  void* get(const void* stream, Alloc alloc, Wait wait) {
    ++clock;
    Slot* s = nullptr;
    for (int i = 0; i < n && !s; ++i)
      if (slot[i].stream == stream) s = &slot[i];
    if (!s) {
      if (n < SLOTS) {
        s = &slot[n++];
      } else {
        s = &slot[0];
        for (Slot& o : slot)
          if (o.used < s->used) s = &o;
        if (clock - s->used < IDLE || !wait()) return nullptr;
      }
      s->stream = stream;
    }
    s->used = clock;
    if (!s->ptr && (s->tried == 0 || clock - s->tried >= IDLE)) {
      s->tried = clock;
      s->ptr = alloc();
    }
    return s->ptr;
  }

  // Gives every workspace back through free_(ptr); the caller has waited for the device.
  template <class Free>
  void clear(Free free_) {
    for (int i = 0; i < n; ++i) {
      if (slot[i].ptr) free_(slot[i].ptr);
      slot[i] = Slot{};
    }
    n = 0;
  }
};

}  // namespace mk
