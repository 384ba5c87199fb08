// Host-only pieces of the session runtime that need no GPU: tests compile
// them alone.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <thread>
#include <vector>

namespace tmpm {

// Runs fn(begin, end) over [0, n) in up to 16 host threads (chunks of at
// least min_chunk items; small ranges run inline).  Used for the per-particle
// host work of uploads, admissions and readbacks.  fn may not throw.
template <class F>
void parallel_for(size_t n, F&& fn, size_t min_chunk = 16384) {
  const unsigned hw = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
  const size_t chunks = std::min<size_t>(hw, (n + min_chunk - 1) / min_chunk);
  if (chunks <= 1) {
    fn((size_t)0, n);
    return;
  }
  const size_t step = (n + chunks - 1) / chunks;
  std::vector<std::thread> pool;
  pool.reserve(chunks);
  size_t inline_from = chunks;  // chunks no thread could be started for run here
  for (size_t c = 1; c < chunks; ++c) {
    const size_t b = c * step, e = std::min(n, b + step);
    if (b >= e) break;
    try {
      pool.emplace_back([&fn, b, e] { fn(b, e); });
    } catch (...) {
      inline_from = c;
      break;
    }
  }
  fn((size_t)0, std::min(n, step));
  for (size_t c = inline_from; c < chunks; ++c)
    if (c * step < n) fn(c * step, std::min(n, c * step + step));
  for (auto& t : pool) t.join();
}

// ---------------------------------------------------------------------------
// Readback of a plain session: records to world
// ---------------------------------------------------------------------------
constexpr size_t kRecordFloats = 29;  // x, v and volume, C, F, plastic state of a particle, as the device lays them out

// The columns of a world that a readback writes.
template <class Column>
struct StateColumns {
  Column pos, vel, F, C, force, plastic;
};

// Particles [first, first + count) of `w` after a readback, into `to`, which
// may be w's own columns (gpu.rs:2295-2329 apply_gpu_transfers): f32 widened
// to f64.  Forces are one-shot; fixed particles end with zero v and C
// (world.rs:419-430).  rec null: there are no records, nothing moved.
template <class World, class Plastic>
void widen_records(const World& w, const StateColumns<double*>& to, const float* rec, size_t first, size_t count,
                   bool plastic, Plastic&& is_plastic) {
  parallel_for(count, [&](size_t b, size_t e) {
    for (size_t k = b; k < e; ++k) {
      const size_t i = first + k;
      for (int q = 0; q < 3; ++q) to.force[3 * i + q] = 0.0;
      if (rec && w.enabled[i] && !w.fixed[i]) {
        const float* r = rec + k * kRecordFloats;
        for (int q = 0; q < 3; ++q) {
          to.pos[3 * i + q] = r[q];
          to.vel[3 * i + q] = r[4 + q];
        }
        for (int q = 0; q < 9; ++q) {
          to.C[9 * i + q] = r[8 + q];
          to.F[9 * i + q] = r[17 + q];
        }
        if (plastic) {
          const bool own = is_plastic(w.material[i]);
          for (int q = 0; q < 3; ++q) to.plastic[3 * i + q] = own ? (double)r[26 + q] : w.plastic[3 * i + q];
        }
        continue;
      }
      const bool still = w.enabled[i] && w.fixed[i];
      for (int q = 0; q < 3; ++q) {
        to.pos[3 * i + q] = w.pos[3 * i + q];
        to.vel[3 * i + q] = still ? 0.0 : w.vel[3 * i + q];
        if (plastic) to.plastic[3 * i + q] = w.plastic[3 * i + q];
      }
      for (int q = 0; q < 9; ++q) {
        to.C[9 * i + q] = still ? 0.0 : w.C[9 * i + q];
        to.F[9 * i + q] = w.F[9 * i + q];
      }
    }
  });
}

// The records of all `n` particles of `w`, which come in pieces of `per`:
// fetch(k, rec) waits for piece k and gives its records (null: there are none)
// and a status.  A status other than 0 ends the readback and leaves the world
// as it was: a single piece is written in place after its status is known,
// several go to `spare`, kept for the next readback, whose columns become the
// world's once all pieces are there.
template <class World, class Column, class Plastic, class Fetch>
int read_pieces(World& w, StateColumns<Column>& spare, size_t n, size_t per, bool plastic, Plastic&& is_plastic,
                Fetch&& fetch) {
  const size_t pieces = std::max<size_t>(1, (n + per - 1) / per);
  StateColumns<double*> to{w.pos.data(), w.vel.data(), w.F.data(), w.C.data(), w.force.data(), w.plastic.data()};
  if (pieces > 1) {
    auto room = [](Column& c, size_t m) {
      if (c.size() != m) c.resize(m);
      return c.data();
    };
    to = {room(spare.pos, 3 * n), room(spare.vel, 3 * n), room(spare.F, 9 * n), room(spare.C, 9 * n),
          room(spare.force, 3 * n), plastic ? room(spare.plastic, 3 * n) : nullptr};
  }
  for (size_t k = 0; k < pieces; ++k) {
    const float* rec = nullptr;
    const int st = fetch(k, rec);
    if (st != 0) return st;
    widen_records(w, to, rec, k * per, std::min(n - k * per, per), plastic, is_plastic);
  }
  if (pieces > 1) {
    w.pos.swap(spare.pos);
    w.vel.swap(spare.vel);
    w.F.swap(spare.F);
    w.C.swap(spare.C);
    w.force.swap(spare.force);
    if (plastic) w.plastic.swap(spare.plastic);
  }
  return 0;
}

}  // namespace tmpm
