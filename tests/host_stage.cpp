// Checks of HostStage without a device: copies are memcpy, "pinned" memory is what
// Fake::pinned names, and calls can be told to fail.
#include "host_stage.hpp"

#include <cstdio>
#include <cstdlib>
#include <string>

struct Fake
{
  using Error = int;
  struct Handle
  {
    int id;
    explicit operator bool() const { return id != 0; }
  };
  struct Stream
  {
  };
  using Event = Handle;
  static constexpr Error ok = 0;
  static inline const char *pinned = nullptr;
  static inline size_t pinned_bytes = 0;
  static inline int allocs = 0, frees = 0, events = 0, direct = 0, staged = 0;
  static inline int max_allocs = 1 << 20, max_events = 1 << 20;
  static inline char *buffer = nullptr;
  static inline size_t buffer_bytes = 0;
  static void reset() { allocs = frees = events = direct = staged = 0; }
  static bool in(const void *p, const char *q, size_t n)
  {
    return q && static_cast<const char *>(p) >= q && static_cast<const char *>(p) < q + n;
  }
  static bool pageable(const void *p) { return !in(p, pinned, pinned_bytes); }
  static Error copy(void *dst, const void *src, size_t n, Stream)
  {
    ++(in(dst, buffer, buffer_bytes) ? staged : direct);
    if (bad_copy-- == 0) return 3;
    std::memcpy(dst, src, n);
    return ok;
  }
  static inline int bad_copy = -1, bad_record = -1, bad_event = -1, waits = 0;  // calls that fail, from 0
  static Error wait(Stream)
  {
    ++waits;
    return ok;
  }
  static Error record(Event, Stream) { return bad_record-- == 0 ? 5 : ok; }
  static Error wait(Event e) { return e.id == bad_event ? 7 : ok; }
  static Error alloc(void **p, size_t n)
  {
    if (allocs >= max_allocs) return 2;
    ++allocs;
    *p = buffer = static_cast<char *>(std::malloc(n));
    buffer_bytes = n;
    return ok;
  }
  static void free(void *p)
  {
    ++frees;
    buffer = nullptr;
    std::free(p);
  }
  static Error create(Event *e)
  {
    if (events >= max_events) return 2;
    *e = {++events};
    return ok;
  }
  static void destroy(Event) { --events; }
  static void clear_error() {}
};

using Stage = pdrd::HostStage<Fake>;

#define CHECK(x)                                               \
  do {                                                         \
    if (!(x)) {                                                \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);      \
      return 1;                                                \
    }                                                          \
  } while (0)

static std::vector<char> data(size_t n)
{
  std::vector<char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = static_cast<char>(i * 2654435761u >> 13);
  return v;
}

// every size around the pieces and groups arrives, through the pieces
static int sizes()
{
  Stage s;
  s.user(true);
  const size_t p = Stage::kPiece, g = p * Stage::kPieces;
  {
    char a = 1, b = 0;
    CHECK(s.copy(0, {}, &b, &a, 1) == Fake::ok && b == 1);  // (the first small copy makes no pieces)
  }
  for (size_t n : {size_t(0), size_t(1), p - 1, p, p + 1, 3 * p, g - 1, g, g + 1, 2 * g + 7}) {
    const std::vector<char> a = data(n);
    std::vector<char> b(n, 0);
    Fake::direct = 0;
    CHECK(s.copy(0, {}, b.data(), a.data(), n) == Fake::ok);
    CHECK(a == b);
  }
  CHECK(Fake::direct == 0 && Fake::staged > 0);
  // another device's copies go directly
  const std::vector<char> a = data(5000);
  std::vector<char> b(5000, 0);
  CHECK(s.copy(1, {}, b.data(), a.data(), a.size()) == Fake::ok && a == b && Fake::direct == 1);
  s.user(false);
  CHECK(Fake::allocs == Fake::frees && Fake::events == 0);
  return 0;
}

// pinned memory of the caller takes the copy directly, from any address in it
static int pinned()
{
  Stage s;
  s.user(true);
  const size_t n = 3 * Stage::kPiece + 5;
  const std::vector<char> a = data(n);
  std::vector<char> b(n + 64, 0);
  Fake::pinned = b.data();
  Fake::pinned_bytes = b.size();
  for (size_t off : {size_t(0), size_t(64)}) {
    Fake::reset();
    CHECK(s.copy(0, {}, b.data() + off, a.data(), n) == Fake::ok);
    CHECK(std::memcmp(b.data() + off, a.data(), n) == 0);
    CHECK(Fake::direct == 1 && Fake::staged == 0 && Fake::allocs == 0);
  }
  s.user(false);
  return 0;
}

// one small copy makes no buffer, a second one does without events; a copy of several
// pieces makes both at once; the last user takes them along
static int made_late()
{
  const size_t p = Stage::kPiece;
  const std::vector<char> a = data(3 * p);
  std::vector<char> b(3 * p, 0);
  Stage s;
  for (int round = 0; round < 2; ++round) {
    Fake::reset();
    s.user(true);
    CHECK(s.copy(0, {}, b.data(), a.data(), 100) == Fake::ok);
    CHECK(Fake::allocs == 0 && Fake::events == 0 && Fake::direct == 1);
    CHECK(s.copy(0, {}, b.data(), a.data(), 100) == Fake::ok);
    CHECK(Fake::allocs == 1 && Fake::events == 0 && Fake::direct == 1 && Fake::staged == 1);
    CHECK(s.copy(0, {}, b.data(), a.data(), 3 * p) == Fake::ok && a == b);
    CHECK(Fake::allocs == 1 && Fake::events == Stage::kPieces && Fake::direct == 1);
    s.user(false);
    CHECK(Fake::frees == 1 && Fake::events == 0);
  }
  Fake::reset();
  s.user(true);
  CHECK(s.copy(0, {}, b.data(), a.data(), 3 * p) == Fake::ok);
  CHECK(Fake::allocs == 1 && Fake::events == Stage::kPieces && Fake::direct == 0);
  s.user(false);
  // a buffer or an event that cannot be had: directly, and nothing is left over
  for (int *limit : {&Fake::max_allocs, &Fake::max_events}) {
    Fake::reset();
    *limit = limit == &Fake::max_events ? 3 : 0;
    std::fill(b.begin(), b.end(), 0);
    s.user(true);
    CHECK(s.copy(0, {}, b.data(), a.data(), 3 * p) == Fake::ok && a == b && Fake::direct == 1);
    CHECK(Fake::allocs == Fake::frees && Fake::events == 0);
    s.user(false);
    *limit = 1 << 20;
  }
  return 0;
}

// a call that fails in the middle of a group ends the copy with its error, and not
// before the stream is empty: the pieces are the next copy's
static int failures()
{
  const size_t n = 5 * Stage::kPiece;
  const std::vector<char> a = data(n);
  std::vector<char> b(n, 0);
  Stage s;
  s.user(true);
  for (int which = 0; which < 3; ++which) {
    Fake::waits = 0;
    (which == 0 ? Fake::bad_copy : which == 1 ? Fake::bad_record : Fake::bad_event) = 2;
    CHECK(s.copy(0, {}, b.data(), a.data(), n) == (which == 0 ? 3 : which == 1 ? 5 : 7));
    CHECK(Fake::waits == 1);
    Fake::bad_copy = Fake::bad_record = Fake::bad_event = -1;
    CHECK(s.copy(0, {}, b.data(), a.data(), n) == Fake::ok && a == b);
  }
  s.user(false);
  return 0;
}

int main(int argc, char **argv)
{
  const std::string name = argc > 1 ? argv[1] : "";
  if (name == "sizes") return sizes();
  if (name == "pinned") return pinned();
  if (name == "made_late") return made_late();
  if (name == "failures") return failures();
  return 2;
}
