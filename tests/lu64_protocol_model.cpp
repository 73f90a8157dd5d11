// Host model of the FP64 LU-SGS sweeps' hand-offs (test infrastructure:
// compiled and run by tests/test_lu64_protocol_model.py on the CPU, also
// under ThreadSanitizer; nothing of the library links it).
//
// What is modelled: the forward and the backward sweep of k_lu_sweep64
// (turns2d_urans_git_amd/csrc/ot2d_kernels.hip), scalar,
//   forward   s(c,k) = (f + sv (A(c-1,k) s(c-1,k) + B(c,k-1) s(c,k-1))) di
//   backward  s(c,k) = f - sv (A'(c+1,k) s(c+1,k) + B'(c,k+1) s(c,k+1)) di
// over the columns c = 0 .. ni+1, where the halo columns (sv = 0, di = 1)
// return their f.  The rows are cut into W blocks of R; the halo row above is
// a row of the last block where that has room.  A workgroup is
//   the computing wave   row r of the block does column t - r at step t; reads
//                        its slots two steps ahead, again if a tag was stale;
//                        publishes `consumed` at every third slot
//   NP producers         records of step t into ring slot t % S
//   the mail wave        the fill of the block's first row: windows of WIN
//                        columns of the upstream block's edge row (the ready
//                        prefix of each poll), or the halo row's records; it
//                        applies the row's B itself, and sets a tag of its own
// Results are two words per value, {low, sweep} and {high, sweep}, stored one
// after the other; a reader takes an entry only when both carry its sweep.
// Workgroups take their block from a ticket of their direction.  The ring's
// records and fills are plain memory, so ThreadSanitizer checks the hand-offs;
// a slot whose tag is stale is not read (the kernel reads it and drops it).
//
// Checks, per sweep: every result equals a sequential evaluation in the same
// operation order, bit for bit; every wait ends (BoundedWait).  Exit status 0
// when all hold, 1 otherwise.
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <random>
#include <string>
#include <thread>
#include <vector>

#include "ot2d_plain.h"

namespace {

struct Cfg {
  int ni = 21, nk = 11, R = 4, S = 6, NP = 2, WIN = 4;
  int nsweep = 30, streams = 3, ninst = 2;
  int xcds = 2, slots = 3;        // CU slots per XCD, shared by all streams
  bool plant_ring_bug = false;    // refill a slot one step early (TSan must flag it)
  bool plant_half_entry = false;  // take an entry by its first word alone
  unsigned seed = 1;
};

thread_local std::mt19937 rng_tl{12345};
void jitter(int pct) {
  if ((int)(rng_tl() % 100) < pct) {
    if (rng_tl() % 4 == 0) std::this_thread::sleep_for(std::chrono::microseconds(rng_tl() % 60));
    else std::this_thread::yield();
  }
}

uint64_t bits(double d) { uint64_t u; std::memcpy(&u, &d, 8); return u; }
double val(uint64_t u) { double d; std::memcpy(&d, &u, 8); return d; }

struct Cell { double f, sv, di, A, B; };   // A, B: applied to the cell's own s for its neighbours

// one instance: cells (c, k) with c = 0 .. ni+1, k = -1 .. nk (halo rows)
struct Instance {
  int ni, nk, R, W, TD;
  std::vector<Cell> fwd, bwd;             // f of bwd unused (the forward result)
  std::vector<std::atomic<uint64_t>> H[2];   // forward, backward results: two words per (block, step, row)
  std::atomic<uint64_t> ticket[2];
  Instance(int ni_, int nk_, int R_) : ni(ni_), nk(nk_), R(R_), W((nk_ + R_ - 1) / R_), TD(ni_ + 2 + R_ - 1) {
    for (int d = 0; d < 2; ++d) {
      H[d] = std::vector<std::atomic<uint64_t>>((size_t)W * TD * R * 2);
      for (auto& h : H[d]) h.store(0);
      ticket[d].store(0);
    }
    fwd.resize((size_t)(ni + 2) * (nk + 2));
    bwd.resize(fwd.size());
  }
  Cell& at(int dir, int c, int k) { return (dir > 0 ? fwd : bwd)[(size_t)(k + 1) * (ni + 2) + c]; }
  std::atomic<uint64_t>* word(int dir, int w, int step, int r) {
    return &H[dir > 0 ? 0 : 1][(((size_t)w * TD + step) * R + r) * 2];
  }
  double result(int dir, int w, int step, int r) {
    std::atomic<uint64_t>* p = word(dir, w, step, r);
    return val((p[0].load() & 0xffffffffull) | (p[1].load() << 32));
  }
};

struct Counts { std::atomic<long> sweeps{0}, wrong{0}, timeouts{0}; };

struct Ring {
  int R;
  std::vector<Cell> rec;      // [S][R]
  std::vector<double> fill;   // [S]
  std::vector<std::atomic<int>> tag_rec, tag_fill;
  std::atomic<int> consumed{0}, abort{0};
  Ring(int S, int R_) : R(R_), rec((size_t)S * R_), fill(S, 0.0), tag_rec(S), tag_fill(S) {
    for (int i = 0; i < S; ++i) { tag_rec[i].store(0); tag_fill[i].store(0); }
  }
};

template <typename Ready>
bool wait_until(Ready ready, Ring& rg) {
  ot2d::BoundedWait wait;
  wait.start();
  while (!ready()) {
    if (rg.abort.load(std::memory_order_relaxed)) return false;
    if (wait.over()) {
      rg.abort.store(1);
      return false;
    }
    std::this_thread::yield();
  }
  return true;
}

void run_workgroup(const Cfg& cfg, Instance& I, int dir, Counts& cnt) {
  const uint64_t n = I.ticket[dir > 0 ? 0 : 1].fetch_add(1, std::memory_order_relaxed);
  const int wb = (int)(n % (uint64_t)I.W);
  const uint32_t tag = (uint32_t)(n / (uint64_t)I.W) + 1u;
  const int R = cfg.R, S = cfg.S, NP = cfg.NP, ni = I.ni;
  const int w = dir > 0 ? wb : I.W - 1 - wb;
  const int left = I.nk - R * w, nr = left >= R ? R : left + 1, NT = ni + 1 + nr;
  const bool from_block = dir > 0 ? w > 0 : w < I.W - 1;
  const bool has_in = from_block || dir > 0 || left == R;
  Ring rg(S, R);
  if (!has_in)
    for (auto& t : rg.tag_fill) t.store(INT32_MAX);
  // record of row r at the block's step t (outside the grid: zero)
  auto rec_of = [&](int t, int r) -> Cell {
    const int st = dir > 0 ? t : NT - 1 - t, c = st - r, k = R * w + r;
    if (c < 0 || c > ni + 1 || k > I.nk || (k == I.nk && (I.nk % R == 0 || c == 0 || c == ni + 1)))
      return Cell{0, 0, 0, 0, 0};
    Cell x = I.at(dir, c, k);
    if (dir < 0) {
      // the forward result of this record step
      std::atomic<uint64_t>* p = I.word(1, w, st, r);
      x.f = val((p[0].load(std::memory_order_relaxed) & 0xffffffffull) | (p[1].load(std::memory_order_relaxed) << 32));
    }
    return x;
  };
  std::vector<std::thread> th;
  for (int p = 0; p < NP; ++p)
    th.emplace_back([&, p] {
      rng_tl.seed(cfg.seed * 1000003u + (unsigned)(w * 131 + p * 7 + dir));
      for (int t = p; t < NT; t += NP) {
        jitter(20);
        std::vector<Cell> v(R);
        for (int r = 0; r < R; ++r) v[r] = rec_of(t, r);
        const int need = cfg.plant_ring_bug ? t - S : t - S + 1;
        if (!wait_until([&] { return rg.consumed.load(std::memory_order_acquire) >= need; }, rg)) return;
        for (int r = 0; r < R; ++r) rg.rec[(size_t)(t % S) * R + r] = v[r];
        rg.tag_rec[t % S].store(t + 1, std::memory_order_release);
      }
    });
  if (has_in)
    th.emplace_back([&] {
      rng_tl.seed(cfg.seed * 65537u + (unsigned)(w * 37 + dir));
      auto deliver = [&](int t1, int m, const double* b) -> bool {
        for (int i = 0; i < m; ++i) {
          const int te = t1 + i;
          if (!wait_until([&] { return rg.consumed.load(std::memory_order_acquire) >= te - S + 1; }, rg)) return false;
          rg.fill[te % S] = b[i];
          rg.tag_fill[te % S].store(te + 1, std::memory_order_release);
        }
        return true;
      };
      const std::vector<double> zero(cfg.WIN, 0.0);
      auto col = [&](int e) { return dir > 0 ? e + 1 : ni - e; };
      const int kup = dir > 0 ? R * w - 1 : R * w + R;   // the upstream row
      bool ok = deliver(0, 1, zero.data());
      for (int e0 = 0; e0 < ni && ok; e0 += cfg.WIN) {
        const int ne = ni - e0 < cfg.WIN ? ni - e0 : cfg.WIN;
        std::vector<double> b(cfg.WIN);
        if (!from_block) {
          for (int i = 0; i < ne; ++i) b[i] = I.at(dir, col(e0 + i), kup).B * I.at(dir, col(e0 + i), kup).f;
          ok = deliver(e0 + 1, ne, b.data());
          continue;
        }
        const int wn = w - dir, re = dir > 0 ? R - 1 : 0;
        ot2d::BoundedWait wait;
        wait.start();
        for (int done = 0; done < ne && ok;) {
          jitter(10);
          // one poll: the ready prefix of the window
          std::vector<uint64_t> x0(cfg.WIN), x1(cfg.WIN);
          int ready = 0;
          for (int i = 0; i < ne; ++i) {
            std::atomic<uint64_t>* p = I.word(dir, wn, col(e0 + i) + re, re);
            x0[i] = p[0].load(std::memory_order_relaxed);
            x1[i] = p[1].load(std::memory_order_relaxed);
          }
          while (ready < ne && (uint32_t)(x0[ready] >> 32) == tag &&
                 (cfg.plant_half_entry || (uint32_t)(x1[ready] >> 32) == tag))
            ++ready;
          if (ready <= done) {
            if (rg.abort.load() || wait.over()) {
              rg.abort.store(1);
              ok = false;
            }
            std::this_thread::yield();
            continue;
          }
          wait.start();
          for (int i = done; i < ready; ++i)
            b[i] = I.at(dir, col(e0 + i), kup).B * val((x0[i] & 0xffffffffull) | (x1[i] << 32));
          ok = deliver(e0 + 1 + done, ready - done, b.data() + done);
          done = ready;
        }
      }
      for (int t = ni + 1; t < NT && ok; ++t) ok = deliver(t, 1, zero.data());
    });
  // the computing wave
  {
    rng_tl.seed(cfg.seed * 7919u + (unsigned)(w * 17 + dir));
    struct Read { std::vector<Cell> rec; double fill = 0; bool fresh = false; };
    Read q[3];
    auto rd = [&](int t, Read& x) {
      const int s = t % S;
      x.fresh = rg.tag_rec[s].load(std::memory_order_acquire) >= t + 1 &&
                rg.tag_fill[s].load(std::memory_order_acquire) >= t + 1;
      if (!x.fresh) return;
      x.rec.assign(rg.rec.begin() + (size_t)s * R, rg.rec.begin() + (size_t)(s + 1) * R);
      x.fill = rg.fill[s];
    };
    std::vector<double> T(R, 0.0), B(R, 0.0), s(R);
    bool ok = true;
    rd(0, q[0]);
    if (NT > 1) rd(1, q[1]);
    for (int t = 0; t < NT && ok; ++t) {
      jitter(10);
      Read& C = q[t % 3];
      if (!C.fresh) {
        ok = wait_until([&] {
          return rg.tag_rec[t % S].load(std::memory_order_acquire) >= t + 1 &&
                 rg.tag_fill[t % S].load(std::memory_order_acquire) >= t + 1;
        }, rg);
        if (!ok) break;
        rd(t, C);
      }
      if (t % S % 3 == 2) rg.consumed.store(t + 1, std::memory_order_release);
      if (t + 2 < NT) rd(t + 2, q[(t + 2) % 3]);
      const int first = dir > 0 ? 0 : R - 1;
      for (int r = 0; r < R; ++r) {
        const double b = r == first ? C.fill : B[r - dir];
        const Cell& x = C.rec[r];
        s[r] = dir > 0 ? (x.f + x.sv * (T[r] + b)) * x.di : x.f - x.sv * (T[r] + b) * x.di;
      }
      const int st = dir > 0 ? t : NT - 1 - t;
      for (int r = 0; r < R; ++r) {
        T[r] = C.rec[r].A * s[r];
        B[r] = C.rec[r].B * s[r];
        std::atomic<uint64_t>* p = I.word(dir, w, st, r);
        const uint64_t u = bits(s[r]), tg = (uint64_t)tag << 32;
        p[0].store(tg | (u & 0xffffffffull), std::memory_order_relaxed);
        if (r == 0 || r == R - 1) jitter(15);
        p[1].store(tg | (u >> 32), std::memory_order_relaxed);
      }
    }
    if (!ok) cnt.timeouts++;
  }
  for (auto& x : th) x.join();
}

struct Dispatcher {
  std::mutex mu;
  std::condition_variable cv;
  std::vector<int> free_slots;
  Dispatcher(int nx, int slots) : free_slots(nx, slots) {}
  void acquire(int x) {
    std::unique_lock<std::mutex> g(mu);
    cv.wait(g, [&] { return free_slots[x] > 0; });
    --free_slots[x];
  }
  void release(int x) {
    { std::lock_guard<std::mutex> g(mu); ++free_slots[x]; }
    cv.notify_all();
  }
};

// the two sweeps in sequence; s(c, k) for k = -1 .. nk
void sequential(Instance& I, std::vector<double>& sf, std::vector<double>& sb) {
  const int nc = I.ni + 2;
  auto ix = [&](int c, int k) { return (size_t)(k + 1) * nc + c; };
  sf.assign((size_t)nc * (I.nk + 2), 0.0);
  for (int k = -1; k <= I.nk; ++k)
    for (int c = 0; c < nc; ++c) sf[ix(c, k)] = I.at(1, c, k).f;
  for (int k = 0; k < I.nk; ++k)
    for (int c = 1; c <= I.ni; ++c) {
      const Cell& x = I.at(1, c, k);
      const double T = I.at(1, c - 1, k).A * sf[ix(c - 1, k)], b = I.at(1, c, k - 1).B * sf[ix(c, k - 1)];
      sf[ix(c, k)] = (x.f + x.sv * (T + b)) * x.di;
    }
  sb = sf;
  for (int k = I.nk - 1; k >= 0; --k)
    for (int c = I.ni; c >= 1; --c) {
      const Cell& x = I.at(-1, c, k);
      const double T = I.at(-1, c + 1, k).A * sb[ix(c + 1, k)], b = I.at(-1, c, k + 1).B * sb[ix(c, k + 1)];
      sb[ix(c, k)] = sf[ix(c, k)] - x.sv * (T + b) * x.di;
    }
}

void run_stream(const Cfg& cfg, int sid, Dispatcher& disp, std::atomic<int>& base_at, Counts& cnt) {
  std::vector<std::unique_ptr<Instance>> inst;
  for (int i = 0; i < cfg.ninst; ++i) inst.emplace_back(new Instance(cfg.ni, cfg.nk - i, cfg.R));
  std::mt19937 r(cfg.seed * 31u + (unsigned)sid);
  std::uniform_real_distribution<double> U(-1, 1), P(0.05, 0.45);
  for (int sw = 0; sw < cfg.nsweep; ++sw) {
    std::vector<std::vector<double>> sf(cfg.ninst), sb(cfg.ninst);
    for (int i = 0; i < cfg.ninst; ++i) {
      Instance& I = *inst[i];
      for (int k = -1; k <= I.nk; ++k)
        for (int c = 0; c <= I.ni + 1; ++c) {
          const bool in = c > 0 && c <= I.ni && k >= 0 && k < I.nk;
          I.at(1, c, k) = Cell{U(r), in ? 0.5 : 0.0, in ? 0.5 + P(r) : 1.0, P(r), P(r)};
          I.at(-1, c, k) = I.at(1, c, k);
          I.at(-1, c, k).A = P(r);
          I.at(-1, c, k).B = P(r);
        }
      sequential(I, sf[i], sb[i]);
    }
    for (int dir : {1, -1}) {
      // grid (W, instances): linear workgroup n goes to XCD (base + n) % xcds,
      // each XCD dispatching in order
      const int wmax = inst[0]->W, base = base_at.fetch_add(wmax * cfg.ninst);
      std::vector<std::vector<std::pair<int, int>>> q(cfg.xcds);
      for (int i = 0; i < cfg.ninst; ++i)
        for (int x = 0; x < wmax; ++x) q[(base + i * wmax + x) % cfg.xcds].emplace_back(i, x);
      std::vector<std::thread> xt;
      for (int x = 0; x < cfg.xcds; ++x)
        xt.emplace_back([&, x] {
          std::vector<std::thread> wg;
          for (auto& e : q[x]) {
            disp.acquire(x);
            wg.emplace_back([&, x, e] {
              if (e.second < inst[e.first]->W) run_workgroup(cfg, *inst[e.first], dir, cnt);
              disp.release(x);
            });
          }
          for (auto& t : wg) t.join();
        });
      for (auto& t : xt) t.join();
      for (int i = 0; i < cfg.ninst; ++i) {
        Instance& I = *inst[i];
        const std::vector<double>& want = dir > 0 ? sf[i] : sb[i];
        for (int k = 0; k < I.nk; ++k)
          for (int c = 1; c <= I.ni; ++c) {
            const int w = k / I.R, row = k % I.R;
            if (bits(I.result(dir, w, c + row, row)) != bits(want[(size_t)(k + 1) * (I.ni + 2) + c])) cnt.wrong++;
          }
      }
    }
    cnt.sweeps++;
  }
}

}  // namespace

int main(int argc, char** argv) {
  Cfg cfg;
  for (int i = 1; i < argc; ++i) {
    const std::string a = argv[i];
    auto num = [&](const char* k) { return a.rfind(k, 0) == 0 ? std::atoi(a.c_str() + std::strlen(k)) : -1; };
    if (a == "--plant-ring-bug") cfg.plant_ring_bug = true;
    else if (a == "--plant-half-entry") cfg.plant_half_entry = true;
    else if (num("--sweeps=") >= 0) cfg.nsweep = num("--sweeps=");
    else if (num("--streams=") >= 0) cfg.streams = num("--streams=");
    else if (num("--slots=") >= 0) cfg.slots = num("--slots=");
    else if (num("--xcds=") >= 0) cfg.xcds = num("--xcds=");
    else if (num("--nk=") >= 0) cfg.nk = num("--nk=");
    else if (num("--ni=") >= 0) cfg.ni = num("--ni=");
    else if (num("--seed=") >= 0) cfg.seed = (unsigned)num("--seed=");
    else {
      std::fprintf(stderr, "unknown argument %s\n", a.c_str());
      return 2;
    }
  }
  if (cfg.S % 3 != 0 || cfg.nk < cfg.ninst + 1) return 2;
  Dispatcher disp(cfg.xcds, cfg.slots);
  Counts cnt;
  std::atomic<int> base{0};
  std::vector<std::thread> st;
  for (int s = 0; s < cfg.streams; ++s) st.emplace_back([&, s] { run_stream(cfg, s, disp, base, cnt); });
  for (auto& t : st) t.join();
  std::printf("sweeps=%ld wrong=%ld timeouts=%ld\n", cnt.sweeps.load(), cnt.wrong.load(), cnt.timeouts.load());
  return cnt.wrong == 0 && cnt.timeouts == 0 ? 0 : 1;
}
