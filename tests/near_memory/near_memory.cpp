// The near store's host side (rigidfibers_amd/csrc/rf_store.h) on a model of the device memory.
#include <cstdio>
#include <cstdlib>
#include <set>

#include "rf_store.h"

#define CHECK(c)                                                    \
  do {                                                              \
    if (!(c)) {                                                     \
      std::printf("line %d: %s does not hold\n", __LINE__, #c);     \
      std::exit(1);                                                 \
    }                                                               \
  } while (0)

struct Model {
  static std::set<void*> live;
  static bool full;
  static int device, placed;  // the thread's current GPU, and the last allocation's
  static int current_device() { return device; }
  static bool make_current(int d) {
    device = d;
    return d < 2;
  }
  static void* allocate(long bytes) {
    if (full) return nullptr;
    CHECK(live.empty());  // the old store has been given back
    void* p = std::malloc(bytes);
    placed = device;
    live.insert(p);
    return p;
  }
  static void release(void* p) {
    CHECK(live.erase(p) == 1);
    std::free(p);
  }
};
std::set<void*> Model::live;
bool Model::full = false;
int Model::device = 0, Model::placed = -1;

int main() {
  {
    rf::NearMemory<Model> m;
    CHECK(!m.holds_system() && m.bytes() == 0);  // before any assembly
    CHECK(m.reserve(100) && !m.holds_system() && m.bytes() == 400);
    m.begin();
    CHECK(!m.holds_system());
    m.complete();
    CHECK(m.holds_system());
    // an assembly that outgrows the store and finds no memory
    m.begin();
    Model::full = true;
    CHECK(!m.reserve(1000));
    CHECK(!m.holds_system() && m.data() == nullptr && m.capacity() == 0 && Model::live.empty());
    // and the next one, which finds some
    Model::full = false;
    m.begin();
    CHECK(m.reserve(1000) && m.data() != nullptr && !m.holds_system());
    m.complete();
    CHECK(m.holds_system() && m.capacity() == 1000);
    // growing voids what was stored, also outside an assembly
    CHECK(m.reserve(2000) && !m.holds_system());
  }
  CHECK(Model::live.empty());
  for (int own = 0; own < 2; ++own) {
    // the store of GPU `own` grows in a thread whose current GPU is the other
    rf::NearMemory<Model> m;
    m.set_device(own);
    for (int caller = 0; caller < 2; ++caller) {
      Model::device = caller;
      CHECK(m.reserve(10) && Model::placed == own && Model::device == caller);
      Model::full = true;
      CHECK(!m.reserve(20) && Model::device == caller);
      Model::full = false;
    }
  }
  CHECK(Model::live.empty());
  std::puts("ok");
  return 0;
}
