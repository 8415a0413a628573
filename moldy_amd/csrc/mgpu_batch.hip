// Many independent systems (replicas of uneven size) stepped together, and
// the autotuner that picks launch shapes and the schedule.  No counterpart
// in the reference, which runs one system per process.
//
// Each replica is an ordinary engine with its own stream and device buffers.
// Schedules:
//   MGPU_SCHED_GRAPH          one hipGraph holds one MD step of every
//                             replica as parallel branches (fork/join
//                             events); a step of the whole set is one
//                             hipGraphLaunch;
//   MGPU_SCHED_STREAM_GRAPHS  each replica replays its own step graph on its
//                             own stream, round robin;
//   MGPU_SCHED_STREAMS        eager launches, round robin over the streams;
//   MGPU_SCHED_GROUPED        one launch per stage for all replicas: each
//                             replica's step is recorded (kernel, shape,
//                             parameters) instead of launched, the records
//                             are merged into grouped launches (the replica
//                             found from the block index, its parameters from
//                             a table), and those launches are captured in
//                             one graph.
// The autotuner first times each engine's tunable launch shapes on its own
// force evaluation (pure: no state changes), then times the schedules over a
// few MD steps and keeps the fastest.
#include "mgpu_internal.h"

#include <algorithm>
#include <array>
#include <chrono>
#include <map>
#include <tuple>

using namespace mgpu;

struct mgpu_batch {
   int device = 0;
   hipStream_t origin = nullptr;
   std::vector<mgpu_engine *> eng;
   hipGraph_t graph = nullptr;
   hipGraphExec_t exec = nullptr;
   std::vector<int> cap_version, cap_precision;
   unsigned long cap_epoch = 0;
   std::vector<hipEvent_t> ev;          // [0] fork, [1] done, then one per engine
   int schedule = MGPU_SCHED_GRAPH;
   std::string err;
   // grouped schedule: the merged launches of one step, their parameter
   // tables on the device, and the graph that holds them
   struct Group {
      void (*launch)(const GroupTab &, unsigned, unsigned, size_t, hipStream_t);
      GroupTab tab;
      unsigned grid, block;
      size_t shm;
   };
   std::vector<Group> groups;
   long recorded = 0;                   // the replicas' own launches in one step, summed
   DBuf<char> d_gtab;
   hipGraph_t ggraph = nullptr;
   hipGraphExec_t gexec = nullptr;
   std::vector<int> gcap_version, gcap_precision;
   unsigned long gcap_epoch = 0;
   bool grouped_ok = false;             // groups, table and graph are built
   void *pin = nullptr;                 // pinned host staging of the replicas' records and flags
   size_t pin_bytes = 0;
};

namespace {

template <class F> int bguard(mgpu_batch *b, F &&f) {
   if (!b) return MGPU_E_ARG;
   try {
      return f();
   } catch (const HipError &h) {
      b->err = std::string("HIP error ") + hipGetErrorString(h.err) + " in " + h.what;
      return MGPU_E_HIP;
   } catch (const StatusError &s) {
      b->err = s.msg;
      return s.code;
   }
}

void drop_branch_graph(mgpu_batch *b) {
   if (b->exec) (void)hipGraphExecDestroy(b->exec);
   if (b->graph) (void)hipGraphDestroy(b->graph);
   b->exec = nullptr;
   b->graph = nullptr;
}

void drop_grouped(mgpu_batch *b) {
   if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
   if (b->ggraph) (void)hipGraphDestroy(b->ggraph);
   b->gexec = nullptr;
   b->ggraph = nullptr;
   b->groups.clear();
   b->grouped_ok = false;
}

void drop_graph(mgpu_batch *b) {
   drop_branch_graph(b);
   drop_grouped(b);
}

bool graph_stale(const mgpu_batch *b) {
   if (!b->exec || b->cap_epoch != g_alloc_epoch || b->cap_version.size() != b->eng.size()) return true;
   for (size_t r = 0; r < b->eng.size(); r++)
      if (b->cap_version[r] != b->eng[r]->geom_version || b->cap_precision[r] != b->eng[r]->precision) return true;
   return false;
}

bool grouped_stale(const mgpu_batch *b) {
   if (!b->grouped_ok || b->gcap_epoch != g_alloc_epoch || b->gcap_version.size() != b->eng.size()) return true;
   for (size_t r = 0; r < b->eng.size(); r++)
      if (b->gcap_version[r] != b->eng[r]->geom_version || b->gcap_precision[r] != b->eng[r]->precision) return true;
   return false;
}

void ensure_events(mgpu_batch *b) {
   while (b->ev.size() < b->eng.size() + 2) {
      hipEvent_t e;
      HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      b->ev.push_back(e);
   }
}

// One step of every replica captured as parallel branches of one graph.
void capture_batch(mgpu_batch *b) {
   drop_branch_graph(b);
   ensure_events(b);
   unsigned long epoch = g_alloc_epoch;
   HIPCHK(hipStreamBeginCapture(b->origin, hipStreamCaptureModeThreadLocal));
   try {
      HIPCHK(hipEventRecord(b->ev[0], b->origin));
      for (size_t r = 0; r < b->eng.size(); r++) {
         mgpu_engine *e = b->eng[r];
         HIPCHK(hipStreamWaitEvent(e->stream, b->ev[0], 0));
         e->capturing = true;
         md_step_launch(e);
         e->capturing = false;
         HIPCHK(hipEventRecord(b->ev[2 + r], e->stream));
         HIPCHK(hipStreamWaitEvent(b->origin, b->ev[2 + r], 0));
      }
   } catch (...) {
      for (auto *e : b->eng) e->capturing = false;
      hipGraph_t g = nullptr;
      (void)hipStreamEndCapture(b->origin, &g);
      if (g) (void)hipGraphDestroy(g);
      throw;
   }
   HIPCHK(hipStreamEndCapture(b->origin, &b->graph));
   if (epoch != g_alloc_epoch) throw StatusError{MGPU_E_STATE, "allocation during batch graph capture"};
   HIPCHK(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
   b->cap_epoch = g_alloc_epoch;
   b->cap_version.clear();
   b->cap_precision.clear();
   for (auto *e : b->eng) {
      b->cap_version.push_back(e->geom_version);
      b->cap_precision.push_back(e->precision);
   }
}

// One step of replica e recorded instead of launched, with the
// real/reciprocal overlap off (one stream).  A first pass only makes the
// buffers of that layout (their allocation, and the clearing of fresh
// memory, run for real; the records are dropped).  The second pass runs
// under a stream capture that is thrown away, so a launch that does not
// record (a kernel without a grouped form, a copy) runs nowhere and shows up
// as a node of that graph: then the step cannot be grouped and the result
// is empty.
std::vector<LaunchRec> record_step(mgpu_engine *e) {
   std::vector<LaunchRec> recs;
   const int ov = e->overlap;
   e->overlap = 0;
   auto undo = [&]() {
      e->rec = nullptr;
      e->capturing = false;
      e->overlap = ov;
   };
   try {
      e->rec = &recs;
      e->capturing = true;   // no timing events
      md_step_launch(e);
   } catch (...) {
      undo();
      throw;
   }
   recs.clear();
   const unsigned long epoch = g_alloc_epoch;
   HIPCHK(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
   e->capturing = true;
   try {
      md_step_launch(e);
   } catch (...) {
      undo();
      hipGraph_t g = nullptr;
      (void)hipStreamEndCapture(e->stream, &g);
      if (g) (void)hipGraphDestroy(g);
      throw;
   }
   undo();
   hipGraph_t g = nullptr;
   HIPCHK(hipStreamEndCapture(e->stream, &g));
   size_t nodes = 0;
   const hipError_t rc = hipGraphGetNodes(g, nullptr, &nodes);
   (void)hipGraphDestroy(g);
   HIPCHK(rc);
   if (nodes || epoch != g_alloc_epoch) recs.clear();
   return recs;
}

// Whether every launch of e's step has a grouped form: all but the FP64
// Ewald sum and the surface-dipole glue do.  The first recording pass runs
// outside any capture, so a step with a launch that does not record must
// be refused here, before it is recorded (that launch would run for real);
// the captured second pass only confirms it.
bool groupable(const mgpu_engine *e) {
   return (e->alpha <= 1e-7 || e->precision == MGPU_MIXED) && !e->surface_dipole;
}

// Merge the replicas' records into grouped launches.  Each replica's
// launches stay in its own order; at every stage one kernel at the heads of
// the replicas' lists is launched for all of them (a greedy common
// supersequence that lets a list wait for a kernel it holds further on),
// so replicas whose steps differ by a launch or two (an extra weight table,
// a force-partial sum) still share the other stages.
// Parameters and block starts go to one device table; the launches are
// captured in one graph on the batch's stream.
void build_grouped(mgpu_batch *b) {
   drop_grouped(b);
   const size_t R = b->eng.size();
   std::vector<std::vector<LaunchRec>> rec(R);
   // (a replica's first recording pass may allocate; its second may not)
   b->recorded = 0;
   for (size_t r = 0; r < R; r++) {
      rec[r] = record_step(b->eng[r]);
      b->recorded += (long)rec[r].size();
      if (rec[r].empty()) throw StatusError{MGPU_E_STATE, "replica " + std::to_string(r) + ": a launch of its step "
                                                          "has no grouped form"};
   }
   struct Pending {
      size_t first;                       // table offset of the parameters
      size_t start;                       // table offset of the block starts
      int n, stride;
      const LaunchRec *proto;
      unsigned grid;
      size_t shm;
   };
   std::vector<Pending> pend;
   std::vector<char> host;
   auto take = [&](size_t bytes) {
      const size_t o = (host.size() + 255) & ~(size_t)255;
      host.resize(o + bytes);
      return o;
   };
   std::vector<size_t> head(R, 0);
   using Key = std::pair<const void *, unsigned>;
   for (;;) {
      // Of the (kernel, block) pairs at the heads of the lists, take one
      // that no list still holds further on (a list that needs it later
      // would need a launch of its own), the one at the most heads; only
      // when every head is held further on, the one at the most heads.  Of
      // equal counts, the one that reached its count first in replica order.
      std::map<Key, int> votes;
      std::vector<Key> order;
      for (size_t r = 0; r < R; r++) {
         if (head[r] >= rec[r].size()) continue;
         const LaunchRec &h = rec[r][head[r]];
         if (votes[{h.key, h.block}]++ == 0) order.push_back({h.key, h.block});
      }
      if (order.empty()) break;
      std::map<Key, bool> later;
      for (size_t r = 0; r < R; r++)
         for (size_t i = head[r] + 1; i < rec[r].size(); i++) {
            const Key k{rec[r][i].key, rec[r][i].block};
            if (votes.count(k)) later[k] = true;
         }
      Key best{nullptr, 0};
      int bestv = 0;
      for (int pass = 0; pass < 2 && !bestv; pass++)
         for (const Key &k : order)
            if ((pass == 1 || !later.count(k)) && votes[k] > bestv) {
               bestv = votes[k];
               best = k;
            }
      std::vector<const LaunchRec *> mem;
      for (size_t r = 0; r < R; r++) {
         if (head[r] >= rec[r].size()) continue;
         const LaunchRec &h = rec[r][head[r]];
         if (h.key != best.first || h.block != best.second) continue;
         head[r]++;
         if (h.grid) mem.push_back(&h);
      }
      if (mem.empty()) continue;
      Pending p{};
      p.n = (int)mem.size();
      p.stride = (int)((mem[0]->args.size() + 15) & ~(size_t)15);
      p.proto = mem[0];
      p.first = take((size_t)p.n * p.stride);
      for (int m = 0; m < p.n; m++) {
         if (mem[m]->args.size() != mem[0]->args.size()) throw StatusError{MGPU_E_STATE, "grouped records disagree"};
         memcpy(host.data() + p.first + (size_t)m * p.stride, mem[m]->args.data(), mem[m]->args.size());
      }
      p.start = take(sizeof(int) * (p.n + 1));
      int *st = (int *)(host.data() + p.start);
      long long g = 0;
      for (int m = 0; m < p.n; m++) {
         st[m] = (int)g;
         g += mem[m]->grid;
         p.shm = std::max(p.shm, mem[m]->shm);
      }
      if (g > 0x7fffffff) throw StatusError{MGPU_E_CAPACITY, "grouped launch larger than one grid"};
      st[p.n] = (int)g;
      p.grid = (unsigned)g;
      pend.push_back(p);
   }
   b->d_gtab.reserve(host.size());
   HIPCHK(hipMemcpy(b->d_gtab.p, host.data(), host.size(), hipMemcpyHostToDevice));
   for (const Pending &p : pend) {
      mgpu_batch::Group gr;
      gr.launch = p.proto->launch;
      gr.tab.args = (uint64_t)(uintptr_t)(b->d_gtab.p + p.first);
      gr.tab.start = (const int *)(b->d_gtab.p + p.start);
      gr.tab.n = p.n;
      gr.tab.stride = p.stride;
      gr.grid = p.grid;
      gr.block = p.proto->block;
      gr.shm = p.shm;
      b->groups.push_back(gr);
   }
   HIPCHK(hipStreamBeginCapture(b->origin, hipStreamCaptureModeThreadLocal));
   try {
      for (const auto &gr : b->groups) gr.launch(gr.tab, gr.grid, gr.block, gr.shm, b->origin);
   } catch (...) {
      hipGraph_t g = nullptr;
      (void)hipStreamEndCapture(b->origin, &g);
      if (g) (void)hipGraphDestroy(g);
      throw;
   }
   HIPCHK(hipStreamEndCapture(b->origin, &b->ggraph));
   HIPCHK(hipGraphInstantiate(&b->gexec, b->ggraph, nullptr, nullptr, 0));
   b->gcap_epoch = g_alloc_epoch;
   b->gcap_version.clear();
   b->gcap_precision.clear();
   for (auto *e : b->eng) {
      b->gcap_version.push_back(e->geom_version);
      b->gcap_precision.push_back(e->precision);
   }
   b->grouped_ok = true;
}

// Enqueue nsteps of every replica under schedule s (no host sync).
void enqueue_steps(mgpu_batch *b, int nsteps, bool init_h0, int s) {
   if (s == MGPU_SCHED_GROUPED)
      for (size_t r = 0; r < b->eng.size(); r++)
         if (!groupable(b->eng[r]))
            throw StatusError{MGPU_E_ARG, "replica " + std::to_string(r) +
                                              ": FP64 Ewald and surface-dipole steps have no grouped launches"};
   for (auto *e : b->eng) {
      md_load_cell(e);
      md_reset_record(e, nsteps, init_h0);
      zero_async(e, e->d_iflags.p, sizeof(int) * 48);
   }
   if (nsteps <= 0) return;
   // The first step runs eagerly (it makes every buffer, and is what a profile
   // times) unless the schedule's captured step is current: then every step
   // is a replay.
   bool prof = false;
   for (auto *e : b->eng) prof = prof || e->prof_on;
   const bool replay_all = !prof && ((s == MGPU_SCHED_GROUPED && !grouped_stale(b)) ||
                                     (s == MGPU_SCHED_GRAPH && !graph_stale(b)));
   const int first = replay_all ? 0 : 1;
   if (!replay_all) {
      for (auto *e : b->eng) md_step_launch(e);
      if (nsteps == 1) return;
   }
   if (s == MGPU_SCHED_GROUPED) {
      if (grouped_stale(b)) build_grouped(b);
      ensure_events(b);
      for (size_t r = 0; r < b->eng.size(); r++) {
         HIPCHK(hipEventRecord(b->ev[2 + r], b->eng[r]->stream));
         HIPCHK(hipStreamWaitEvent(b->origin, b->ev[2 + r], 0));
      }
      for (int k = first; k < nsteps; k++) HIPCHK(hipGraphLaunch(b->gexec, b->origin));
      HIPCHK(hipEventRecord(b->ev[1], b->origin));
      for (auto *e : b->eng) HIPCHK(hipStreamWaitEvent(e->stream, b->ev[1], 0));
   } else if (s == MGPU_SCHED_GRAPH) {
      if (graph_stale(b)) capture_batch(b);
      ensure_events(b);
      for (size_t r = 0; r < b->eng.size(); r++) {
         HIPCHK(hipEventRecord(b->ev[2 + r], b->eng[r]->stream));
         HIPCHK(hipStreamWaitEvent(b->origin, b->ev[2 + r], 0));
      }
      for (int k = first; k < nsteps; k++) HIPCHK(hipGraphLaunch(b->exec, b->origin));
      HIPCHK(hipEventRecord(b->ev[1], b->origin));
      for (auto *e : b->eng) HIPCHK(hipStreamWaitEvent(e->stream, b->ev[1], 0));
   } else if (s == MGPU_SCHED_STREAM_GRAPHS) {
      for (auto *e : b->eng) ensure_step_graph(e);
      for (int k = 1; k < nsteps; k++)
         for (auto *e : b->eng) HIPCHK(hipGraphLaunch(e->graph_exec, e->stream));
   } else {
      for (int k = 1; k < nsteps; k++)
         for (auto *e : b->eng) md_step_launch(e);
   }
}

// Every replica's record and flags come back through one pinned host
// buffer: the copies are all enqueued before any is waited for (copies into
// pageable memory would each wait for their own).
void finish(mgpu_batch *b, int nsteps, double *trace) {
   const size_t R = b->eng.size();
   const size_t tw = (trace && nsteps > 0) ? (size_t)md_trace_width() * nsteps : 0;
   const size_t per = tw * sizeof(double) + 48 * sizeof(int);   // one replica's record, then its flags
   if (b->pin_bytes < R * per) {
      if (b->pin) (void)hipHostFree(b->pin);
      b->pin = nullptr;
      b->pin_bytes = 0;
      HIPCHK(hipHostMalloc(&b->pin, R * per, hipHostMallocDefault));
      b->pin_bytes = R * per;
   }
   char *pin = (char *)b->pin;
   for (size_t r = 0; r < R; r++) {
      mgpu_engine *e = b->eng[r];
      if (tw) HIPCHK(hipMemcpyAsync(pin + r * per, e->d_trace.p, sizeof(double) * tw, hipMemcpyDeviceToHost, e->stream));
      HIPCHK(hipMemcpyAsync(pin + r * per + tw * sizeof(double), e->d_iflags.p, sizeof(int) * 41,
                            hipMemcpyDeviceToHost, e->stream));
   }
   for (auto *e : b->eng) HIPCHK(hipStreamSynchronize(e->stream));
   for (size_t r = 0; r < R; r++) {
      if (tw) memcpy(trace + r * tw, pin + r * per, sizeof(double) * tw);
      int fl[41];
      memcpy(fl, pin + r * per + tw * sizeof(double), sizeof fl);
      try {
         handle_flags(b->eng[r], fl);
      } catch (const StatusError &s) {
         throw StatusError{s.code, "replica " + std::to_string(r) + ": " + s.msg};
      }
   }
}

// Process-wide memory of tuned shapes: (precision, nrows, lmax, nsites/4096,
// gridded sum) -> (S(k) workgroups, MFMA back-projection partitions, FP64
// partitions, overlap).
std::map<std::tuple<int, int, int, int, bool>, std::array<int, 4>> g_tuned;

}  // namespace

// Time the tunable launch shapes of e's force evaluation and keep the
// fastest: the S(k) workgroup count and the back-projection row partitions
// of the MFMA Ewald (mixed precision), or the row partitions of the FP64
// back-projection; none of these where the gridded sum runs, which has no such
// shape (only the overlap is tuned then).  Results are identical up to the
// summation order of partial sums.
void mgpu::autotune_engine(mgpu_engine *e, int reps, int *sk_blocks, int *npart) {
   if (e->alpha <= 1e-7) return;
   const bool grid = grid_chosen(e);
   auto key = std::make_tuple(e->precision, e->nrows, e->lmax, e->nsites / 4096, grid);
   auto it = g_tuned.find(key);
   if (it != g_tuned.end()) {
      if (!grid) {
         e->tune_sk_blocks = it->second[0];
         e->tune_force_parts = it->second[1];
         e->tune_npart = it->second[2];
      }
      e->overlap = it->second[3];
   } else {
      hipEvent_t t0, t1;
      HIPCHK(hipEventCreate(&t0));
      HIPCHK(hipEventCreate(&t1));
      const bool prof = e->prof_on;
      e->prof_on = false;
      int nrep = reps;
      auto time_eval = [&]() {
         e->geom_version++;   // re-plan with the new shape
         eval_forces_device(e, true);
         HIPCHK(hipEventRecord(t0, e->stream));
         for (int k = 0; k < nrep; k++) eval_forces_device(e, true);
         HIPCHK(hipEventRecord(t1, e->stream));
         HIPCHK(hipEventSynchronize(t1));
         float ms = 0;
         HIPCHK(hipEventElapsedTime(&ms, t0, t1));
         return ms;
      };
      // coordinate descent over one shape at a time; workgroup targets in
      // whole rounds of the resident slots
      // two passes over the candidates, each scored by its faster pass, so
      // that a clock ramp or a neighbour's burst does not pick the shape
      auto tune = [&](int &field, const std::vector<int> &cand, int passes = 2) {
         std::vector<float> t(cand.size(), 1e30f);
         for (int pass = 0; pass < passes; pass++)
            for (size_t c = 0; c < cand.size(); c++) {
               field = cand[c];
               t[c] = std::min(t[c], time_eval());
            }
         field = cand[std::min_element(t.begin(), t.end()) - t.begin()];
      };
      if (!grid && e->precision == MGPU_MIXED) {
         const int slots = e->ncu;   // one S(k) workgroup per CU (LDS)
         tune(e->tune_sk_blocks, {2 * slots, 3 * slots, 4 * slots, 6 * slots, 8 * slots, 12 * slots});
         tune(e->tune_force_parts, {0, 1, 2, 4});
      } else if (!grid) {
         tune(e->tune_npart, {4, 8, 16, 32});
      }
      // real space beside the Ewald sum, or after it: a difference of a few
      // per cent, so longer trials and more passes than the shapes above
      nrep = std::max(reps, 10);
      tune(e->overlap, {1, 0}, 4);
      e->prof_on = prof;
      (void)hipEventDestroy(t0);
      (void)hipEventDestroy(t1);
      g_tuned[key] = {e->tune_sk_blocks, e->tune_force_parts, e->tune_npart, e->overlap};
   }
   e->geom_version++;
   if (sk_blocks) *sk_blocks = !grid && e->precision == MGPU_MIXED ? e->tune_sk_blocks : 0;
   if (npart) *npart = grid ? 0 : e->precision == MGPU_MIXED ? e->tune_force_parts : e->tune_npart;
}

extern "C" {

int mgpu_batch_create(mgpu_batch **bp, int device) {
   if (!bp) return MGPU_E_ARG;
   *bp = nullptr;
   mgpu_batch *b = new mgpu_batch();
   b->device = device;
   int rc = bguard(b, [&] {
      HIPCHK(hipSetDevice(device));
      HIPCHK(hipStreamCreateWithFlags(&b->origin, hipStreamNonBlocking));
      return 0;
   });
   if (rc) {
      delete b;
      return rc;
   }
   *bp = b;
   return 0;
}

void mgpu_batch_destroy(mgpu_batch *b) {
   if (!b) return;
   (void)hipSetDevice(b->device);
   if (b->origin) (void)hipStreamSynchronize(b->origin);
   drop_graph(b);
   b->d_gtab.free();
   if (b->pin) (void)hipHostFree(b->pin);
   for (auto ev : b->ev) (void)hipEventDestroy(ev);
   if (b->origin) (void)hipStreamDestroy(b->origin);
   delete b;
}

const char *mgpu_batch_last_error(const mgpu_batch *b) { return b ? b->err.c_str() : "null batch"; }

int mgpu_batch_add(mgpu_batch *b, mgpu_engine *e) {
   return bguard(b, [&] {
      if (!e || !e->have_dyn || e->n_full == 0) {
         b->err = "engine needs mgpu_set_dynamics, mgpu_upload_state and mgpu_upload_momenta";
         return (int)MGPU_E_STATE;
      }
      if (e->device != b->device) {
         b->err = "engine on another device";
         return (int)MGPU_E_ARG;
      }
      if (e->dyn_const_pressure) {
         b->err = "a barostat engine re-plans its cell every step: run it with mgpu_md_steps";
         return (int)MGPU_E_ARG;
      }
      b->eng.push_back(e);
      drop_graph(b);
      return 0;
   });
}

int mgpu_batch_steps(mgpu_batch *b, int nsteps, int init_h0, int schedule, double *trace) {
   return bguard(b, [&] {
      if (nsteps < 0 || b->eng.empty()) {
         b->err = "no engines or nsteps < 0";
         return (int)MGPU_E_ARG;
      }
      HIPCHK(hipSetDevice(b->device));
      const int s = schedule < 0 ? b->schedule : schedule;
      enqueue_steps(b, nsteps, init_h0 != 0, s);
      finish(b, nsteps, trace);
      return 0;
   });
}

int mgpu_batch_grouped_plan(const mgpu_batch *b, long out[2]) {
   if (!b || !out) return MGPU_E_ARG;
   if (!b->grouped_ok) return MGPU_E_STATE;
   out[0] = (long)b->groups.size();
   out[1] = b->recorded;
   return 0;
}

int mgpu_batch_autotune(mgpu_batch *b, int trial_steps, int *schedule, double ms_per_step[4]) {
   return bguard(b, [&] {
      if (b->eng.empty() || trial_steps < 2) {
         b->err = "no engines or fewer than 2 trial steps";
         return (int)MGPU_E_ARG;
      }
      HIPCHK(hipSetDevice(b->device));
      for (auto *e : b->eng) autotune_engine(e, 3, nullptr, nullptr);
      // each schedule with the engines' own real/reciprocal stream overlap
      // and with it off (replicas already run side by side)
      std::vector<int> own;
      for (auto *e : b->eng) own.push_back(e->overlap);
      auto set_overlap = [&](bool off) {
         for (size_t r = 0; r < b->eng.size(); r++) {
            const int want = off ? 0 : own[r];
            if (b->eng[r]->overlap != want) {
               b->eng[r]->overlap = want;
               b->eng[r]->geom_version++;   // captured graphs follow the stream layout
            }
         }
         drop_graph(b);
      };
      constexpr int NS = 4;
      bool grouped = true;
      for (auto *e : b->eng) grouped = grouped && groupable(e);
      double t[2][NS];
      for (int off = 0; off < 2; off++) {
         set_overlap(off);
         for (int s = 0; s < NS; s++) {
            // the grouped step records with the overlap off: timed once
            if (s == MGPU_SCHED_GROUPED && (!grouped || !off)) {
               t[off][s] = 1e30;
               continue;
            }
            // warm up outside the timing with as many steps as the trial,
            // so that the trial's record buffers and captured step are ready
            enqueue_steps(b, trial_steps, false, s);
            finish(b, trial_steps, nullptr);
            HIPCHK(hipDeviceSynchronize());
            auto t0 = std::chrono::steady_clock::now();
            enqueue_steps(b, trial_steps, false, s);
            finish(b, trial_steps, nullptr);
            auto t1 = std::chrono::steady_clock::now();
            t[off][s] = std::chrono::duration<double, std::milli>(t1 - t0).count() / trial_steps;
         }
      }
      int best = 0;
      for (int k = 1; k < 2 * NS; k++)
         if (t[k / NS][k % NS] < t[best / NS][best % NS]) best = k;
      set_overlap(best / NS);
      b->schedule = best % NS;
      if (schedule) *schedule = best % NS;
      if (ms_per_step)
         for (int s = 0; s < NS; s++) {
            const double m = std::min(t[0][s], t[1][s]);
            ms_per_step[s] = m < 1e29 ? m : -1.0;   // -1: the schedule does not apply
         }
      return 0;
   });
}

int mgpu_autotune(mgpu_engine *e, int reps, int *sk_blocks, int *npart) {
   if (!e) return MGPU_E_ARG;
   try {
      if (!e->have_system || e->n_full == 0) {
         e->err = "mgpu_upload_state not called";
         return MGPU_E_STATE;
      }
      HIPCHK(hipSetDevice(e->device));
      autotune_engine(e, reps < 1 ? 3 : reps, sk_blocks, npart);
      return 0;
   } catch (const HipError &h) {
      e->err = std::string("HIP error ") + hipGetErrorString(h.err) + " in " + h.what;
      return MGPU_E_HIP;
   } catch (const StatusError &s) {
      e->err = s.msg;
      return s.code;
   }
}

}  // extern "C"
