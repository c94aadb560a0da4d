// The scratch memory that contexts keep between calls (Spare, ctx.hpp).
#include <algorithm>
#include <mutex>
#include <vector>

#include "ctx.hpp"

namespace psoci {

namespace {

// Every context's scratch, and which of it is in use: a context's own thread
// takes and leaves it, any thread whose allocation fails may free the rest.
// (Never destroyed: contexts may outlive this file's statics.)
struct Registry {
  std::mutex mu;
  std::vector<Spare*> all;
};
Registry& registry() {
  static Registry* r = new Registry;
  return *r;
}

bool release_idle(Spare& s) {
  bool any = false;
  for (int i = 0; i < 4; ++i)
    if (!s.busy[i] && s.buf[i].p) {
      s.buf[i].release();
      s.allowed = kSpareBytes / 16;
      any = true;
    }
  return any;
}

}  // namespace

Spare::Spare() {
  Registry& r = registry();
  std::lock_guard<std::mutex> lk(r.mu);
  r.all.push_back(this);
}

Spare::~Spare() {
  Registry& r = registry();
  std::lock_guard<std::mutex> lk(r.mu);
  r.all.erase(std::find(r.all.begin(), r.all.end(), this));
}

bool Spare::give_back() {
  std::lock_guard<std::mutex> lk(registry().mu);
  return release_idle(*this);
}

void Spare::take(int first, int count) {
  std::lock_guard<std::mutex> lk(registry().mu);
  std::fill(busy + first, busy + first + count, true);
}

void Spare::leave(int first, int count) {
  std::lock_guard<std::mutex> lk(registry().mu);
  std::fill(busy + first, busy + first + count, false);
  size_t kept = 0, fr = 0, tot = 0;
  for (const auto& b : buf) kept += b.n;
  if (kept <= allowed) return;
  if (kept <= kSpareBytes && hipMemGetInfo(&fr, &tot) == hipSuccess && kept <= fr / 16) {
    allowed = kept;
    return;
  }
  allowed = kSpareBytes / 16;
  for (int i = first; i < first + count; ++i) buf[i].release();
}

bool give_back_spare(bool others) {
  if (!others) return t_spare && t_spare->give_back();
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  Registry& r = registry();
  std::lock_guard<std::mutex> lk(r.mu);
  bool any = false;
  for (Spare* s : r.all)
    if (s->device == dev && release_idle(*s)) any = true;
  return any;
}

}  // namespace psoci
