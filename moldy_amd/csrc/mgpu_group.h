// Grouped launches: one launch of a kernel for many engines (replicas).
//
// A kernel that can be grouped keeps its body in a device function
//     void b_name(int bx, int nbx, P... params)
// that takes its block index and block count from bx and nbx instead of
// blockIdx.x and gridDim.x.  The direct kernel k_name(P...) calls the body
// with (blockIdx.x, gridDim.x).  The grouped kernel k_grouped<b_name, LB>
// takes a table: each member's parameters (packed as the body's parameter
// types) and the start of its block range in the grid.  A block finds its
// member with one ballot over the starts and runs as block blockIdx.x - start
// of that member, with the member's block count.  The arithmetic of every
// block is the direct kernel's, so a grouped launch gives the same bits.
//
// Host side: in record mode (the engine's rec list set) launch sites append
// a LaunchRec (kernel key, launch shape, packed parameters) instead of
// launching; the batch merges the records of its replicas into grouped
// launches.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <type_traits>
#include <utility>
#include <vector>

namespace mgpu {

// A plain nested struct of the parameters, the same layout on host and
// device.
template <class... T> struct Pack;
template <> struct Pack<> {};
template <class H, class... T> struct Pack<H, T...> {
   H h;
   Pack<T...> t;
};

template <int I, class H, class... T> __host__ __device__ __forceinline__ const auto &pget(const Pack<H, T...> &p) {
   if constexpr (I == 0) return p.h;
   else return pget<I - 1>(p.t);
}

template <class PK> struct PackMaker;
template <> struct PackMaker<Pack<>> {
   static Pack<> make() { return {}; }
};
template <class H, class... T> struct PackMaker<Pack<H, T...>> {
   template <class A, class... B> static Pack<H, T...> make(A &&a, B &&...b) {
      Pack<H, T...> p;
      p.h = static_cast<H>(a);
      p.t = PackMaker<Pack<T...>>::make(std::forward<B>(b)...);
      return p;
   }
};

template <class F> struct BodySig;
template <class... P> struct BodySig<void (*)(int, int, P...)> {
   using pack = Pack<std::decay_t<P>...>;
   static constexpr int n = sizeof...(P);
};

struct GroupTab {
   uint64_t args;      // address of [n][stride] packed parameters (an integer: see group_run)
   const int *start;   // [n + 1] first block of each member; start[n] = grid
   int n, stride;
};

// The member whose block range holds block bx: the number of starts past the
// first that are <= bx, 64 starts a ballot.
__device__ __forceinline__ int group_member(const GroupTab &t, int bx) {
   const int lane = threadIdx.x & 63;
   int r = 0;
   for (int c = 0; c < t.n; c += 64) {
      const int q = c + 1 + lane;
      const bool le = q < t.n && t.start[q] <= bx;
      const int k = __popcll(__ballot(le));
      r = c + k;
      if (k < 64) break;
   }
   return __builtin_amdgcn_readfirstlane(r);
}

template <auto Body, class PK, int... I>
__device__ __forceinline__ void group_call(int bx, int nbx, const PK &p, std::integer_sequence<int, I...>) {
   Body(bx, nbx, pget<I>(p)...);
}

// The parameters are read through a constant-address-space pointer made
// from an integer address: the compiler then reads them in place with scalar
// loads, as it reads a direct kernel's arguments.  (A pointer derived from a
// global pointer argument makes the body's by-value parameters into copies
// in scratch memory.)
template <auto Body> __device__ __forceinline__ void group_run(const GroupTab &t) {
   using S = BodySig<decltype(Body)>;
   using PK = typename S::pack;
   typedef __attribute__((address_space(4))) const PK cPK;
   const int bx = blockIdx.x;
   const int r = group_member(t, bx);
   const int lo = t.start[r], hi = t.start[r + 1];
   const PK &p = *(const PK *)(cPK *)(t.args + (uint64_t)r * t.stride);
   group_call<Body>(bx - lo, hi - lo, p, std::make_integer_sequence<int, S::n>{});
}

template <auto Body, int LB> __global__ __launch_bounds__(LB) void k_grouped(GroupTab t) { group_run<Body>(t); }
template <auto Body, int LB, int WPE>
__global__ __launch_bounds__(LB) __attribute__((amdgpu_waves_per_eu(WPE))) void k_grouped_w(GroupTab t) {
   group_run<Body>(t);
}

// One recorded launch of one engine.
struct LaunchRec {
   const void *key;   // the direct kernel
   void (*launch)(const GroupTab &, unsigned grid, unsigned block, size_t shm, hipStream_t s);
   unsigned grid, block;
   size_t shm;
   std::vector<char> args;
};

// Lets kernel take shm bytes of dynamic LDS: past 64 KiB a launch needs the
// limit raised first.
void allow_lds(const void *kernel, size_t shm);

template <auto Body, int LB, int WPE>
void launch_group(const GroupTab &t, unsigned grid, unsigned block, size_t shm, hipStream_t s) {
   if constexpr (WPE > 0) {
      allow_lds((const void *)k_grouped_w<Body, LB, WPE>, shm);
      k_grouped_w<Body, LB, WPE><<<grid, block, shm, s>>>(t);
   } else {
      allow_lds((const void *)k_grouped<Body, LB>, shm);
      k_grouped<Body, LB><<<grid, block, shm, s>>>(t);
   }
}

// Launch K directly, or append the launch to rec.  LB (and WPE) must be the
// direct kernel's launch bounds (and waves per EU), so that the grouped
// kernel compiles to the same code.
template <auto K, auto Body, int LB, int WPE = 0, class... A>
void glaunch(std::vector<LaunchRec> *rec, hipStream_t s, unsigned grid, unsigned block, size_t shm, A &&...args) {
   if (!rec) {
      allow_lds((const void *)K, shm);
      K<<<grid, block, shm, s>>>(std::forward<A>(args)...);
      return;
   }
   using PK = typename BodySig<decltype(Body)>::pack;
   static_assert(std::is_trivially_copyable<PK>::value, "grouped parameters must be trivially copyable");
   const PK p = PackMaker<PK>::make(std::forward<A>(args)...);
   LaunchRec r;
   r.key = (const void *)K;
   r.launch = &launch_group<Body, LB, WPE>;
   r.grid = grid;
   r.block = block;
   r.shm = shm;
   r.args.resize(sizeof(PK));
   memcpy(r.args.data(), &p, sizeof(PK));
   rec->push_back(std::move(r));
}

}  // namespace mgpu
