#include "runspace.hpp"

#include <list>
#include <mutex>

namespace tbsla {
namespace hip {
namespace {

struct IdleSpace {
  const RunSpaces *owner;
  std::unique_ptr<RunSpace> space;
};

// The idle spaces of every matrix, in the order they were given back.  What
// leaves the list is freed by the caller, outside the lock.
struct Idle {
  std::mutex mu;
  std::list<IdleSpace> list;
  std::size_t bytes = 0;

  void move_out(std::list<IdleSpace>::iterator it, std::list<IdleSpace> &to) {
    bytes -= it->space->mem.bytes();
    to.splice(to.end(), list, it);
  }
};

// (never destroyed: matrices may outlive static objects)
Idle &idle() {
  static Idle *const p = new Idle();
  return *p;
}

}  // namespace

std::unique_ptr<RunSpace> RunSpaces::take(std::size_t bytes) {
  std::list<IdleSpace> out;
  {
    Idle &all = idle();
    std::lock_guard<std::mutex> g(all.mu);
    auto best = all.list.end();
    for (auto it = all.list.begin(); it != all.list.end(); ++it)
      if (it->owner == this && it->space->mem.bytes() >= bytes &&
          (best == all.list.end() || it->space->mem.bytes() < best->space->mem.bytes()))
        best = it;
    if (best != all.list.end()) all.move_out(best, out);
  }
  if (!out.empty()) return std::move(out.front().space);
  std::unique_ptr<RunSpace> s(new RunSpace());
  s->mem.reserve(bytes);
  return s;
}

void RunSpaces::give(std::unique_ptr<RunSpace> s) {
  std::list<IdleSpace> drop, mine;
  mine.push_back(IdleSpace{this, std::move(s)});
  const std::size_t bytes = mine.front().space->mem.bytes();
  if (bytes > kIdleBytes) return;
  Idle &all = idle();
  std::lock_guard<std::mutex> g(all.mu);
  all.list.splice(all.list.end(), mine);
  all.bytes += bytes;
  std::size_t count = 0;
  auto least = all.list.end();
  for (auto it = all.list.begin(); it != all.list.end(); ++it)
    if (it->owner == this) {
      count++;
      if (least == all.list.end() || it->space->mem.bytes() < least->space->mem.bytes()) least = it;
    }
  if (count > kIdleSpaces) all.move_out(least, drop);
  while (all.bytes > kIdleBytes) all.move_out(all.list.begin(), drop);
}

RunSpaces::~RunSpaces() {
  std::list<IdleSpace> drop;
  Idle &all = idle();
  std::lock_guard<std::mutex> g(all.mu);
  for (auto it = all.list.begin(); it != all.list.end();) {
    const auto next = std::next(it);
    if (it->owner == this) all.move_out(it, drop);
    it = next;
  }
}

bool drop_idle_memory() {
  std::list<IdleSpace> drop;
  Idle &all = idle();
  std::lock_guard<std::mutex> g(all.mu);
  drop.swap(all.list);
  all.bytes = 0;
  return !drop.empty();
}

}  // namespace hip
}  // namespace tbsla
