// The island resolver (cbz_islands.h) on one world, on the CPU.  The
// workgroup's LDS ends at an inaccessible page, so an access past its end is an
// error here whatever lies there on a device; the fibers' order is the caller's.
#include <hip/hip_runtime.h>
#include <signal.h>
#include <sys/mman.h>

#define CBZ_RESOLVE_INSTANTIATE
namespace cbz {
char* isl_lds;
}
#include "cbz_islands.h"

namespace {
enum { OK = 0, DEADLOCK = -1, STEPS = -2, ACCESS = -3 };
constexpr size_t kStack = 256 << 10, kGuard = 1 << 20;
sigjmp_buf g_back;
void (*g_fn)(void*);
void* g_arg;

void entry() {
  g_fn(g_arg);
  const int me = emu::cur;
  emu::fibers[me].done = true;
  for (emu::Meet* m : {&emu::wave[me >> 6], &emu::block}) {
    --m->alive;
    m->close();
  }
  _longjmp(emu::scheduler, 1);
}

// Runs a fiber to its next meeting point.
void enter(emu::Fiber& f) {
  if (_setjmp(emu::scheduler)) return;
  if (f.begun) _longjmp(f.at, 1);
  f.begun = true;
  setcontext(&f.ctx);
}

// fn(arg) by nt threads; across: a lane of every wave in turn, instead of a
// wave's lanes one after another
int run_block(void (*fn)(void*), void* arg, int nt, bool across, long max_steps) {
  g_fn = fn;
  g_arg = arg;
  const int waves = nt / 64;
  if (int(emu::fibers.size()) < nt) emu::fibers.resize(nt);
  emu::block = emu::Meet{0, nt, 0};
  for (int w = 0; w < waves; ++w) emu::wave[w] = emu::Meet{0, 64, 0};
  for (int i = 0; i < nt; ++i) {
    emu::Fiber& f = emu::fibers[i];
    if (!f.stack) f.stack = (char*)malloc(kStack);
    getcontext(&f.ctx);
    f.ctx.uc_stack.ss_sp = f.stack;
    f.ctx.uc_stack.ss_size = kStack;
    f.ctx.uc_link = nullptr;
    f.begun = f.done = false;
    makecontext(&f.ctx, entry, 0);
  }
  if (sigsetjmp(g_back, 1)) return ACCESS;
  long last = -1;
  for (long step = 0;; ++step) {
    int left = 0;
    for (int q = 0; q < nt; ++q) {
      const int i = across ? (q % waves) * 64 + q / waves : q;
      if (emu::fibers[i].done) continue;
      emu::cur = i;
      threadIdx.x = i;
      enter(emu::fibers[i]);
      left += !emu::fibers[i].done;
    }
    if (left == 0) return OK;
    long rounds = emu::block.round + (nt - left);
    for (int w = 0; w < waves; ++w) rounds += emu::wave[w].round;
    if (rounds == last) return DEADLOCK;
    if (step >= max_steps) return STEPS;
    last = rounds;
  }
}

void on_segv(int) { siglongjmp(g_back, 1); }

using namespace cbz;
template <class R, int T>
struct Block {
  template <int KIND>
  static void of(void* p) {
    isl_block<R, KIND, T>(*(RS<R>*)p);
  }
};

struct World {
  int32_t n, C, kind, mode, f64, across, threads;
  int64_t mult, fixed, log_cap, max_steps;
  double dt;
  void *pos, *quat, *vel, *rot, *inv_mass, *iit_body, *iit_world, *transform, *last_acc, *motion, *flags;
  void *body0, *body1, *point, *normal, *pen, *c2w, *rel, *cvel, *ddv, *fric, *rest, *labels;
  int64_t* iters;  // [2]
  int32_t* left;   // worlds handed to the serial kernel
};

template <class R, int T>
int resolve(const World& q) {
  RS<R> a;
  memset((void*)&a, 0, sizeof a);
  const int n = q.n, C = q.C;
  auto& b = a.b;
  b.n = n;
  b.stride = n;
  b.pos = (R*)q.pos, b.quat = (R*)q.quat, b.vel = (R*)q.vel, b.rot = (R*)q.rot, b.inv_mass = (R*)q.inv_mass;
  b.iit_body = (R*)q.iit_body, b.iit_world = (R*)q.iit_world, b.transform = (R*)q.transform;
  b.last_acc = (R*)q.last_acc, b.motion = (R*)q.motion, b.flags = (uint8_t*)q.flags;
  auto& c = a.c;
  c.cap = C;
  c.body0 = (int32_t*)q.body0, c.body1 = (int32_t*)q.body1;
  c.point = (R*)q.point, c.normal = (R*)q.normal, c.pen = (R*)q.pen, c.c2w = (R*)q.c2w, c.rel = (R*)q.rel;
  c.cvel = (R*)q.cvel, c.ddv = (R*)q.ddv;
  if (q.kind == KIND_MAT) c.fric = (R*)q.fric, c.rest = (R*)q.rest;
  std::vector<R> imp(kImpPlanes * C + 4), rec(16 * C + 4), pos0(3 * n), save(5 * C), snap(21 * n), log_key(q.log_cap + 1);
  auto align16 = [](R* p) { return (R*)((uintptr_t(p) + 15) & ~uintptr_t(15)); };
  c.imp = align16(imp.data()), c.rec = align16(rec.data());
  std::vector<int32_t> off(n), cnt(n), its(n), nrec(n), cls(kIslWords), idx(C), log_j(q.log_cap + 1), log_it(q.log_cap + 1);
  std::vector<int64_t> log(n);
  std::vector<uint8_t> flag(n);
  const int32_t body_off[2] = {0, n}, overflow = 0;
  int32_t left_list[1], wide_list[1], left_count[LEFT_COUNTS] = {};
  int64_t coff = 0, head = 0;
  a.world_cnt = &C, a.world_coff = &coff, a.overflow = &overflow, a.body_off = body_off, a.world_iters = q.iters;
  a.left_list = left_list, a.wide_list = wide_list, a.left_count = left_count;
  a.isl_nb = (n + 15) & ~15;
  a.isl_off = off.data(), a.isl_cnt = cnt.data(), a.isl_its = its.data(), a.isl_nrec = nrec.data();
  a.isl_log = log.data(), a.isl_cls = cls.data(), a.isl_idx = idx.data();
  a.isl_save = save.data(), a.isl_snap = snap.data(), a.isl_flag = flag.data();
  a.log_key = log_key.data(), a.log_j = log_j.data(), a.log_it = log_it.data();
  a.log_head = &head;
  a.log_cap = q.log_cap;
  a.n_worlds = 1;
  a.dt = R(q.dt), a.iter_mult = q.mult, a.iter_fixed = q.fixed, a.mode = q.mode;
  a.pos0 = pos0.data();
  a.labels = (float*)q.labels;
  // LDS, its last byte before the guard
  const size_t lds = isl_lds_bytes<R, T>(a.isl_nb), page = 4096, room = (lds + page - 1) / page * page;
  char* mem = (char*)mmap(nullptr, room + kGuard, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  mprotect(mem + room, kGuard, PROT_NONE);
  isl_lds = mem + room - lds;
  memset(isl_lds, 0xA5, lds);
  struct sigaction on = {}, was;
  on.sa_handler = on_segv;
  sigaction(SIGSEGV, &on, &was);
  typedef Block<R, T> B;
  void (*fn)(void*) = q.kind == KIND_MAT     ? B::template of<KIND_MAT>
                      : q.kind == KIND_LABEL ? B::template of<KIND_LABEL>
                                             : B::template of<KIND_PLAIN>;
  const int rc = run_block(fn, &a, T, q.across, q.max_steps);
  sigaction(SIGSEGV, &was, nullptr);
  munmap(mem, room + kGuard);
  *q.left = left_count[LEFT_WORLDS] + left_count[LEFT_WIDE];
  return rc;
}
}  // namespace

extern "C" int emu_resolve(const World* q) {
  if (q->threads == 128) return q->f64 ? resolve<double, 128>(*q) : resolve<float, 128>(*q);
  return q->f64 ? resolve<double, 256>(*q) : resolve<float, 256>(*q);
}
