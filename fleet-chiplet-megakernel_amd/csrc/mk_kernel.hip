// Persistent decode megakernel for gfx950 (MI355X): one cooperative launch runs
// every decode iteration of every request.  Each iteration walks a static stage
// program; every stage is tiled over all workgroups, with workgroups ordered
// by the XCD they run on so that one die streams one contiguous chunk of a
// weight matrix and shares activations through its own L2.
//
// Replaces, for the decode path, the reference's device runtime
// (include/mirage/persistent_kernel/persistent_kernel.cuh:693-1907: execute_worker,
// execute_scheduler, prepare_next_batch) and its MI300 task kernels
// (include/mirage/persistent_kernel/tasks/mi300/*.cuh).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "mk_types.h"

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Stage descriptors are written once by the host before the first launch and never by the kernel: reading them
// through the constant address space makes every field a scalar load, so shapes, pointers and everything derived
// from them stay in scalar registers and branches on them are scalar branches.
typedef const __attribute__((address_space(4))) MkStage CStage;
typedef const __attribute__((address_space(4))) MkWeight CWeight;

#define MK_SPIN_LIMIT (1u << 24)
#ifndef MK_TUNE_POLL_SLEEP
#define MK_TUNE_POLL_SLEEP 1
#endif

// weight rows in flight per wavefront of the single-token linear (K = 4096 with SwiGLU / K = 4096 plain / K = 12288)
// (a shallow window and more rows parked in LDS across the barrier beat a deep window: whatever a CU has in flight sits in
// front of the control wavefront's barrier poll and input-row loads)
#ifndef MK_TUNE_R8
#define MK_TUNE_R8 2
#endif
#ifndef MK_TUNE_R8N
#define MK_TUNE_R8N 2
#endif
#ifndef MK_TUNE_R4
#define MK_TUNE_R4 2  // K = 2048
#endif
#ifndef MK_TUNE_MOE_M1_R13
#define MK_TUNE_MOE_M1_R13 2  // single-token expert W13: [gate ; up] row pairs in flight per wavefront (K = 2048)
#endif
#ifndef MK_TUNE_MOE_M1_R2
#define MK_TUNE_MOE_M1_R2 1   // single-token expert W2: output rows (x 8 experts) in flight per wavefront
#endif
// multi-token expert linears: cost of a unit's row load relative to one token's reduction (W13 / W2)
#ifndef MK_TUNE_MOE_ROWCOST13
#define MK_TUNE_MOE_ROWCOST13 4
#endif
#ifndef MK_TUNE_MOE_ROWCOST2
#define MK_TUNE_MOE_ROWCOST2 3
#endif
#ifndef MK_TUNE_MOE_M1_PARK
#define MK_TUNE_MOE_M1_PARK 2 // ... and parked in LDS per wavefront while the barrier is awaited
#endif
// units per group of the multi-token expert linears (W13 / W2)
#ifndef MK_TUNE_MOE_R13
#define MK_TUNE_MOE_R13 4
#endif
#ifndef MK_TUNE_MOE_R2
#define MK_TUNE_MOE_R2 16
#endif
#ifndef MK_TUNE_NL
#define MK_TUNE_NL 3
#endif
#ifndef MK_TUNE_W0_KL
#define MK_TUNE_W0_KL 8  // single-token linears with rows of at least this many KB arrive without a workgroup barrier
#endif
#ifndef MK_TUNE_R24
#define MK_TUNE_R24 2
#endif

#if defined(MK_KERNEL_DUAL) || defined(MK_KERNEL_DUAL_PAIR) || defined(MK_KERNEL_DUAL_M1) || defined(MK_KERNEL_DUAL_F32)
#define MK_HAVE_DUAL 1  // ... the dual stages (mk_dual.hip) beside flex, mix and hybrid ones, without latent attention, delta rule and selective scan
#else
#define MK_HAVE_DUAL 0
#endif
#if defined(MK_KERNEL_HYB) || defined(MK_KERNEL_HYB_PAIR) || defined(MK_KERNEL_HYB_M1) || defined(MK_KERNEL_HYB_F32) || MK_HAVE_DUAL
#define MK_HAVE_HYB 1
#else
#define MK_HAVE_HYB 0
#endif
#if defined(MK_KERNEL_MIX) || defined(MK_KERNEL_MIX_PAIR) || defined(MK_KERNEL_MIX_M1) || defined(MK_KERNEL_MIX_F32) || MK_HAVE_HYB
#define MK_HAVE_MIX 1  // this translation unit holds a kernel with the mix stages (mk_mix.hip) beside the flex ones
#else
#define MK_HAVE_MIX 0
#endif

// kernels that run iterations of several portions inside prompts, and nothing else
#if defined(MK_KERNEL_DENSE_PAIR) || defined(MK_KERNEL_FLEX_PAIR) || defined(MK_KERNEL_MIX_PAIR) || defined(MK_KERNEL_HYB_PAIR) || defined(MK_KERNEL_DUAL_PAIR)
#define MK_PAIR 1
#else
#define MK_PAIR 0
#endif

#define MK_NO_LISTS 0x7fffffff
struct Ctx {
  int tid;   // threadIdx.x, made opaque for every stage that runs: see run_stage_program
  CStage *st;  // descriptor of the stage that runs (null before the first one)
  int vid;   // virtual workgroup id: xcd-major, so vids [x*quota, (x+1)*quota) share an L2
  int G;     // workgroups in the grid
  int xcd;   // XCC_ID of the CU this workgroup landed on
  int quota; // workgroups on this XCD
  int nxcd;  // XCDs that received at least one workgroup
  unsigned quotas[8];  // workgroups on each of the first 8 XCD ids (0 = unused)
  int xi;     // index of this XCD among the XCDs in use
  int rank;   // rank of this workgroup inside its XCD
  unsigned epoch;
  bool pending;  // an arrive has been posted that no wait has consumed yet
  bool dead;     // the watchdog fired somewhere: unwind
  long long t_wait;  // (profiling) tick at which the last barrier_wait completed
  int *sh_dead;
  MkSync *sync;
  const int *sh_tok;  // LDS copy of this iteration's token metadata: [0] position, [1] batch slot, [2] first token of the request, [3] first page-table entry
  bool even_xcds;     // every die in use runs the same number of workgroups, so die index = vid / quota
  int *sh_ticket;     // two LDS work counters, used alternately by consecutive executed stages; [2] = seq (multi-token: ~seq) of the
                      // MoE stage that last filled the workgroup's expert list (kept outside the stages' scratch LDS)
  int seq;            // stages executed so far by this workgroup
  unsigned prof_n;    // entries this workgroup has written into the caller's profiler tensor
  bool wrote_through; // the stage that just ran wrote all its outputs with write-through stores: no L2 write-back at its barrier
  bool arrive_w0;     // ... and all of them from wavefront 0, after a workgroup barrier, having reset the next stage's work
                      // counter itself: the arrival then needs no workgroup barrier of its own (see barrier_arrive)
  // A split-K linear whose consumer is a full-row norm leaves its K-slice partials unsummed: the norm stage, which reads
  // every row anyway, sums them (slice order, then the residual, then one rounding: the same arithmetic).
  int defer_S;            // slices left unsummed by the stage that just ran (0: none)
  int defer_rows;         // token rows per slice in the partial buffer
  int defer_n;            // row length of the partial buffer (the producing linear's outputs)
  const float *defer_part;  // [slice][row][n] fp32
  const void *defer_res;  // residual rows of that linear (null: none)
  int defer_ld_res;
#if MK_PAIR
  int defer_stage;         // the linear itself (its residual rows are each portion's own)
  int rows_ahead;          // where the running stage has dealt rows of portions in front already: mk_rows_ahead of them
  int portion;             // that the running stage runs for
  bool keeps_sum;          // the running linear leaves no sum (mk_keeps_sum)
#endif
#if MK_HAVE_MIX
  bool mx_split;  // the latent attention (delta rule) that just ran left some request in chunks (its heads in slices)
#endif
#if MK_HAVE_DUAL
  const int *state_ids;  // MkRuntime::state_ids
#endif
#ifdef MK_TRACE
  long long mark[4];  // (tracing builds) wall-clock marks the running stage sets, stored next to its stage timing
#endif
};
#ifdef MK_TRACE
#define MK_MARK(c, i) ((c).mark[i] = (long long)wall_clock64())
#else
#define MK_MARK(c, i) ((void)0)
#endif

// ----------------------------------------------------------------------------- small helpers
__device__ __forceinline__ float bf_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf_hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }
// round-to-nearest-even float -> bf16 (hardware v_cvt_pk_bf16_f32 on gfx950)
__device__ __forceinline__ uint32_t f2bf(float f) { return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ uint32_t pack2(float a, float b) { return f2bf(a) | (f2bf(b) << 16); }
__device__ __forceinline__ float bfround(float f) { return __uint_as_float(f2bf(f) << 16); }

__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), c, false);
}
__device__ __forceinline__ float dot8(u32x4 a, u32x4 b, float c) {
  c = dot2(a.x, b.x, c);
  c = dot2(a.y, b.y, c);
  c = dot2(a.z, b.z, c);
  c = dot2(a.w, b.w, c);
  return c;
}
// Cross-lane reductions on the DPP path (one VALU instruction per step) instead of LDS-crossbar shuffles: a
// 16-lane row is all-reduced with rotations by 8, 4, 2, 1 (every lane ends with the row total), the four rows of a
// wavefront are then combined through scalar lane reads.  Callers run with whole rows / whole wavefronts active.
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float group16_sum(float v) {
  v += dpp_f32<0x128>(v);  // row_ror:8
  v += dpp_f32<0x124>(v);  // row_ror:4
  v += dpp_f32<0x122>(v);  // row_ror:2
  v += dpp_f32<0x121>(v);  // row_ror:1
  return v;
}
__device__ __forceinline__ float lane_f32(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
__device__ __forceinline__ float wave_sum(float v) {
  v = group16_sum(v);
  return (lane_f32(v, 0) + lane_f32(v, 16)) + (lane_f32(v, 32) + lane_f32(v, 48));
}
// Transposing wavefront reduction: every lane holds partial sums of NV values (NV a power of two <= 16); on return lane
// l holds the wavefront total of value l & (NV - 1).  Stage b pairs the values up and exchanges one of each pair with
// the lane whose bit b differs (one DPP move per pair), so 16 values cost about 50 instructions instead of 16 full
// reductions; the four 16-lane rows are combined with two cross-row permutes at the end.
template <int NV>
__device__ __forceinline__ float transpose_sum(float (&v)[NV], int lane) {
  static_assert(NV == 1 || NV == 2 || NV == 4 || NV == 8 || NV == 16, "power of two");
  if constexpr (NV >= 2) {
    const bool b = lane & 1;
#pragma unroll
    for (int j = 0; j < NV / 2; j++) v[j] = (b ? v[2 * j + 1] : v[2 * j]) + dpp_f32<0xB1>(b ? v[2 * j] : v[2 * j + 1]);  // quad_perm [1,0,3,2]
  }
  if constexpr (NV >= 4) {
    const bool b = lane & 2;
#pragma unroll
    for (int j = 0; j < NV / 4; j++) v[j] = (b ? v[2 * j + 1] : v[2 * j]) + dpp_f32<0x4E>(b ? v[2 * j] : v[2 * j + 1]);  // quad_perm [2,3,0,1]
  }
  if constexpr (NV >= 8) {
    const bool b = lane & 4;
#pragma unroll
    for (int j = 0; j < NV / 8; j++) {
      const float give = b ? v[2 * j] : v[2 * j + 1];
      const float up = dpp_f32<0x104>(give), down = dpp_f32<0x114>(give);  // row_shl:4 (from lane + 4), row_shr:4 (from lane - 4)
      v[j] = (b ? v[2 * j + 1] : v[2 * j]) + (b ? down : up);
    }
  }
  if constexpr (NV >= 16) {
    const bool b = lane & 8;
    v[0] = (b ? v[1] : v[0]) + dpp_f32<0x128>(b ? v[0] : v[1]);  // row_ror:8
  }
  float r = v[0];
  if (NV < 16) r += dpp_f32<0x128>(r);
  if (NV < 8) r += dpp_f32<0x124>(r);
  if (NV < 4) r += dpp_f32<0x122>(r);
  if (NV < 2) r += dpp_f32<0x121>(r);
  r += __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 16) << 2, __builtin_bit_cast(int, r)));
  r += __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __builtin_bit_cast(int, r)));
  return r;
}
__device__ __forceinline__ unsigned xcc_id() {
  // HW_REG_XCC_ID (id 20), bits [3:0]
  return __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 7u;  // MI355X: 8 XCDs
}
__device__ __forceinline__ u32x4 ldg_stream(const u32x4 *p) { return __builtin_nontemporal_load(p); }

// Workgroup barrier behind this wavefront's own LDS accesses and nothing else: where direct-to-LDS requests may be in flight, __syncthreads()
// waits for every load of the wavefront, register loads among them (vmcnt(0) in front of s_barrier), and empties a ring of loads.  Whoever
// requested rows waits for them by count before it comes here.  (The passes of the matrix-core linear: 24576 x 4096 at 64 tokens 41.3 -> 38.5 us,
// 16384 -> 4096 at 8 tokens 27.8 -> 26.4.)
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Loads of data another workgroup produced earlier in this launch.  The per-XCD L2s are write-back and
// not coherent with each other, and the CU's vector L1 is not coherent with anything: producers write back
// their L2 at the barrier (release by the XCD's last arriver), consumers read with device-scope loads
// (sc1: miss the L1, coherent in L2), so no cache invalidate is ever issued.
// (the pointers are cast to the global address space explicitly: an atomic through a generic pointer becomes a flat
// access, which is counted against the LDS queue as well and waits for it)
#define MK_GLOBAL __attribute__((address_space(1)))
__device__ __forceinline__ uint32_t ldc_u32(const void *p) {
  return __hip_atomic_load((const MK_GLOBAL uint32_t *)(unsigned long long)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int ldc_i32(const int *p) { return (int)ldc_u32(p); }
__device__ __forceinline__ float ldc_f32(const float *p) { return __uint_as_float(ldc_u32(p)); }
__device__ __forceinline__ unsigned long long ldc_u64(const void *p) {
  return __hip_atomic_load((const MK_GLOBAL unsigned long long *)(unsigned long long)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u32x4 ldc_16B(const u32x4 *p) {
  const unsigned long long a = ldc_u64(p), b = ldc_u64((const unsigned long long *)p + 1);
  u32x4 r = {(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32)};
  return r;
}
// Sixteen bytes at byte `off` of what a uniform pointer points at, in one request (as two of eight bytes, with the lanes sixteen apart, every
// request carries half of the lines it touches: a row of 4096 summed from four slices, as a norm stage, 7.5 -> 5.4 us; 32-bit 6.0 -> 4.2).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t dev_rows(const void *p) { return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, 0xffffffffu, 0x00027000); }
__device__ __forceinline__ u32x4 ldc_16B(__amdgpu_buffer_rsrc_t rows, int off) { return __builtin_amdgcn_raw_buffer_load_b128(rows, off, 0, 16 /* sc1 */); }
// (They share what they bring through the die's L2 as ordinary loads do: 64 KB of rows into the LDS of every CU in 1.09 us either way, 512 KB in
// 6.4; an acquire in front, which ordinary loads of another workgroup's rows need, takes another 1.8 us and what the L2 held for the next CU
// with it.  So stages of several tokens read rows like this too: dodonex-8b 59.7 -> 57.1 ms, suborax-8b serving 122.2 -> 118.7, 64 streams of
// qwen3-8b 286.2 -> 281.4.)
// Stores that are written through to memory (device scope), for outputs of stages that skip the L2 write-back at
// their barrier.
__device__ __forceinline__ void stc_u16(uint16_t *p, uint16_t v) {
  __hip_atomic_store((__attribute__((address_space(1))) uint16_t *)(unsigned long long)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void stc_f32(float *p, float v) {
  __hip_atomic_store((__attribute__((address_space(1))) unsigned *)(unsigned long long)p, __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void stc_u64(void *p, unsigned long long v) {
  __hip_atomic_store((__attribute__((address_space(1))) unsigned long long *)(unsigned long long)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void stc_i32(int *p, int v) {
  __hip_atomic_store((__attribute__((address_space(1))) int *)(unsigned long long)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// (one store: as two of eight bytes, every 64 bytes of a line had been written through in two requests.  No atomic store is this wide, hence
// the assembly; whoever hands the data over waits for all outstanding stores first.  The s_nop keeps the compiler's next instruction, which
// may write the registers, from following a wide store at once.  qwen3-8b, 64 streams: 300 -> 291 ms, prompt 52.8 -> 50.9 ms.)
__device__ __forceinline__ void stc_16B(u32x4 *p, u32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"((MK_GLOBAL u32x4 *)(unsigned long long)p), "v"(v) : "memory");
}
// four consecutive bf16 outputs of one token row, written through: one 8-byte store when the run is whole and aligned
__device__ __forceinline__ void stc_bf16x4(uint16_t *row, int n0, int n_out, const float (&r)[4]) {
  uint16_t *p = row + n0;
  if (n0 + 3 < n_out && (((unsigned long long)p) & 7) == 0) {
    const unsigned long long v = (unsigned long long)pack2(r[0], r[1]) | ((unsigned long long)pack2(r[2], r[3]) << 32);
    __hip_atomic_store((__attribute__((address_space(1))) unsigned long long *)(unsigned long long)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (n0 + i < n_out) stc_u16(p + i, (uint16_t)f2bf(r[i]));
  }
}
__device__ __forceinline__ uint16_t ldc_half(const uint16_t *p) { return __hip_atomic_load((const MK_GLOBAL uint16_t *)(unsigned long long)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// the same four as 32-bit values (columns behind the row's end: not read)
__device__ __forceinline__ void ldc_bf16x4(const uint16_t *row, int n0, int n_out, float (&r)[4]) {
  const uint16_t *p = row + n0;
  if (n0 + 3 < n_out && (((unsigned long long)p) & 7) == 0) {
    const unsigned long long u = ldc_u64(p);
    r[0] = bf_lo((uint32_t)u);
    r[1] = bf_hi((uint32_t)u);
    r[2] = bf_lo((uint32_t)(u >> 32));
    r[3] = bf_hi((uint32_t)(u >> 32));
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = n0 + i < n_out ? bf2f(ldc_half(p + i)) : 0.f;
  }
}
__device__ __forceinline__ uint16_t ldc_u16(const uint16_t *p) {
  const uintptr_t a = (uintptr_t)p;
  const uint32_t w = ldc_u32((const void *)(a & ~(uintptr_t)3));
  return (uint16_t)((a & 2) ? (w >> 16) : (w & 0xffffu));
}

// ----------------------------------------------------------------------------- grid barrier
// Stage barrier with one arrival counter per XCD (each in 256 bytes of its own, so a die's arrivals meet in that
// die's L2 and only completed lines travel between dies).  Replaces the reference's per-event two-level counters
// (persistent_kernel.cuh:1214-1284).
__device__ __forceinline__ bool spin_ok(MkSync *s, unsigned &spins, unsigned where) {
  ++spins;
  if ((spins & 1023u) == 0) {
    if (__hip_atomic_load(&s->abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
    if (spins >= MK_SPIN_LIMIT) {
      __hip_atomic_store(&s->abort_where, where, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&s->abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
  }
  return true;
}

// arrive: this workgroup's outputs of the current stage are complete: write them back (agent-scope release) and
// count the arrival in the counter of this workgroup's XCD (one line per die, so the 32 arrivals of a die meet
// in that die's L2).  Nothing is returned, so nobody waits on the atomic.
__device__ __forceinline__ void barrier_arrive(Ctx &c) {
  MkSync *s = c.sync;
  if (c.arrive_w0) {
    // Only wavefront 0 has stores outstanding: it waits for them and posts the arrival; the other wavefronts go straight
    // on to the next stage, whose weight prefetch is then in flight while those stores are still being acknowledged
    // (about a microsecond per stage in which the CU otherwise requests nothing).
    c.arrive_w0 = false;
    if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    c.seq++;
    c.epoch++;
    if (threadIdx.x == 0) __hip_atomic_fetch_add(&s->local_ctr[c.xcd][0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    c.wrote_through = false;
    c.pending = true;
    return;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  c.seq++;
  if (threadIdx.x == 0) c.sh_ticket[c.seq & 1] = 0;  // the counter of the stage that starts now (last used two stages ago)
  __syncthreads();
  c.epoch++;
  if (threadIdx.x == 0) {
    if (c.wrote_through) __hip_atomic_fetch_add(&s->local_ctr[c.xcd][0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
      __hip_atomic_fetch_add(&s->local_ctr[c.xcd][0], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
  }
  c.wrote_through = false;
  c.pending = true;
}

// poll (thread 0 only): the barrier is complete when every die's counter has reached quota x epoch.  The eight
// counters are read with independent device-scope loads (one round trip per poll), so completion is seen two hops
// after the last arrival (atomic -> load) instead of going through a leader and a broadcast flag.
__device__ __forceinline__ void barrier_poll(Ctx &c) {
  MkSync *s = c.sync;
  const unsigned epoch = c.epoch;
  unsigned spins = 0;
  unsigned va[8];
  auto issue = [&](unsigned (&v)[8]) {
#pragma unroll
    for (int x = 0; x < 8; x++) v[x] = __hip_atomic_load(&s->local_ctr[x][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  auto done = [&](const unsigned (&v)[8]) -> bool {
    bool ok = true;
#pragma unroll
    for (int x = 0; x < 8; x++) ok = ok && mk_counter_reached(v[x], c.quotas[x] * epoch);
    return ok;
  };
  while (true) {
    issue(va);
    if (done(va) || !spin_ok(s, spins, epoch)) break;
    __builtin_amdgcn_s_sleep(MK_TUNE_POLL_SLEEP);
  }
  *c.sh_dead = (spins >= 1024u) ? (int)__hip_atomic_load(&s->abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
}

// bookkeeping after the workgroup barrier that follows barrier_poll
__device__ __forceinline__ void barrier_done(Ctx &c) {
  c.pending = false;
  c.dead = c.dead || (__builtin_amdgcn_readfirstlane(*c.sh_dead) != 0);
  c.t_wait = (long long)wall_clock64();
}

__device__ __forceinline__ void barrier_wait(Ctx &c) {
  if (!c.pending) return;
  if (threadIdx.x == 0) {
    // The polling wavefront brings the stage's descriptor into the scalar cache: its misses would otherwise follow one another behind the
    // barrier.  (By every wavefront, ahead of the stage, it had held up the requests for weights: a prompt of qwen3-8b 68.0 -> 70.0 ms.)
    typedef const __attribute__((address_space(4))) int CInt;
    CInt *d = (CInt *)c.st;
    static_assert(sizeof(MkStage) == 11 * 64, "one word of every line");
    if (d) asm volatile("" ::"s"(d[0]), "s"(d[16]), "s"(d[32]), "s"(d[48]), "s"(d[64]), "s"(d[80]), "s"(d[96]), "s"(d[112]), "s"(d[128]), "s"(d[144]), "s"(d[160]));
    barrier_poll(c);
  }
  __syncthreads();
  barrier_done(c);
}

// ----------------------------------------------------------------------------- scheduler
// On-GPU continuous batching for offline serving: commit the tokens produced by the previous
// iteration, retire finished requests and recycle their pages, then build the next batch
// (running requests first, then new prefills).  Same observable behaviour on the ten meta
// tensors as the reference's MODE_OFFLINE prepare_next_batch (persistent_kernel.cuh:380-536).
// Runs on one thread.  Returns the number of tokens scheduled.
__device__ __attribute__((noinline)) int mk_prepare_next_batch(const MkRuntime &rt, int *scratch_pages) {
  MkSched *sc = rt.sched;
  const int R = rt.max_requests, B = rt.max_tokens, PS = rt.page_size, NP = rt.max_pages;
  int head = sc->page_queue_head, tail = sc->page_queue_tail;
  // 1. commit outputs of the previous iteration, retire finished requests
  for (int i = 0; i < R; i++) {
    const int req = rt.request_ids[i];
    if (req < 0) continue;
    const int st = rt.step[req];
    const int q0 = rt.qo_indptr[i];
    const int n = rt.qo_indptr[i + 1] - q0;
    const int plen = rt.prompt_lengths[req];
    // a decoding request of a speculating graph keeps what its verify stage accepted: the sampled token of its first
    // row, and one more for every candidate row in front that turned out right (persistent_kernel.cuh:541-552)
    int nc = n;
    if (rt.spec_len > 0 && st >= plen && n > 0) nc = max(1, min(n, ldc_i32(&rt.num_new_tokens[req])));
    for (int j = 0; j < nc; j++) {
      const int pos = st + j + 1;
      if (pos >= plen && pos < rt.max_seq) rt.tokens[(long long)req * rt.max_seq + pos] = rt.output_tokens[q0 + j];
    }
    const int ns = st + nc;
    rt.step[req] = ns;
    const bool full = ns + 1 >= rt.max_seq;
    const bool eos = ns >= plen && rt.tokens[(long long)req * rt.max_seq + ns] == rt.eos_token_id;
    if (full || eos) {
      rt.request_ids[i] = -1;
      const int k0 = rt.kv_indptr[i], k1 = rt.kv_indptr[i + 1];
      for (int j = k0; j < k1; j++) {
        rt.page_queue[tail % NP] = rt.kv_indices[j];
        tail++;
      }
    }
  }
  if (rt.state_ids) {
    // recurrent-state slots move with their requests: the survivors' in front, in order, then the free ones
    int n = 0;
    for (int pass = 0; pass < 2; pass++)
      for (int i = 0; i < R; i++)
        if ((rt.request_ids[i] >= 0) == (pass == 0)) scratch_pages[n++] = rt.state_ids[i];
    for (int i = 0; i < R; i++) rt.state_ids[i] = scratch_pages[i];
  }
  // 2. snapshot the page table (it is compacted in place below)
  const int old_pages = rt.kv_indptr[R];
  for (int i = 0; i < old_pages; i++) scratch_pages[i] = rt.kv_indices[i];
  // 3. running requests keep their slot order; compact over retired slots
  int nreq = 0, ntok = 0, npage = 0;
  bool inner = rt.max_new_per_req > 1;
  for (int i = 0; i < R; i++) {
    const int req = rt.request_ids[i];
    if (req < 0) continue;
    const int k0 = rt.kv_indptr[i];
    const int had = rt.kv_indptr[i + 1] - k0;
    rt.request_ids[nreq] = req;
    rt.qo_indptr[nreq] = ntok;
    rt.kv_indptr[nreq] = npage;
    const int st = rt.step[req];
    int n = rt.prompt_lengths[req] - st;
    if (n > 0) n = min(n, min(rt.max_new_per_req, B - ntok));  // prefill chunk
    else n = min(1 + min(rt.spec_len, min(rt.max_new_per_req - 1, rt.max_seq - 2 - st)), B - ntok);  // decode: the newest token (+ candidate rows,
                                                                                                      // whose ids the n-gram stage fills in)
    inner = inner && (n <= 0 || (st + n < rt.prompt_lengths[req] && st + n + 1 < rt.max_seq));
    for (int j = 0; j < n; j++) {
      rt.input_tokens[ntok + j] = rt.tokens[(long long)req * rt.max_seq + st + j];
      rt.tok_slot[ntok + j] = nreq;
      rt.tok_pos[ntok + j] = st + j;
      rt.tok_first[ntok + j] = ntok;
    }
    const int need = (st + n + PS - 1) / PS;
    const int last = (st + n) % PS;
    rt.kv_last_page_len[nreq] = last == 0 ? PS : last;
    for (int j = 0; j < had; j++) rt.kv_indices[npage + j] = scratch_pages[k0 + j];
    for (int j = had; j < need; j++) {
      rt.kv_indices[npage + j] = rt.page_queue[head % NP];
      head++;
    }
    npage += need;
    ntok += n;
    nreq++;
  }
  // 4. admit new requests while there is room
  while (nreq < R && ntok < B) {
    const int req = sc->next_request_id;
    if (req >= rt.total_requests) break;
    rt.request_ids[nreq] = req;
    rt.qo_indptr[nreq] = ntok;
    rt.kv_indptr[nreq] = npage;
    const int n = min(rt.prompt_lengths[req], min(rt.max_new_per_req, B - ntok));
    inner = inner && n < rt.prompt_lengths[req] && n + 1 < rt.max_seq;
    for (int j = 0; j < n; j++) {
      rt.input_tokens[ntok + j] = rt.tokens[(long long)req * rt.max_seq + j];
      rt.tok_slot[ntok + j] = nreq;
      rt.tok_pos[ntok + j] = j;
      rt.tok_first[ntok + j] = ntok;
    }
    const int need = (n + PS - 1) / PS;
    const int last = n % PS;
    rt.kv_last_page_len[nreq] = last == 0 ? PS : last;
    for (int j = 0; j < need; j++) {
      rt.kv_indices[npage + j] = rt.page_queue[head % NP];
      head++;
    }
    ntok += n;
    npage += need;
    nreq++;
    sc->next_request_id = req + 1;
  }
  // 5. clear unused slots
  for (int i = nreq; i < R; i++) rt.request_ids[i] = -1;
  for (int i = nreq; i <= R; i++) {
    rt.qo_indptr[i] = ntok;
    rt.kv_indptr[i] = npage;
  }
  sc->page_queue_head = head;
  sc->page_queue_tail = tail;
  sc->num_tokens = ntok;
  sc->num_reqs = nreq;
  sc->inner = inner;
  return ntok;
}

// The same step on one wavefront: lane i owns batch slot i (at most 64 slots) in the phases that walk the old batch, and
// candidate request next_request_id + i when new requests are admitted.  What the sequential version carries from slot
// to slot are running sums -- tokens scheduled so far (saturating at the iteration's token budget), pages in the
// compacted table, pages taken from / returned to the ring -- and those are wavefront prefix sums:
//   tokens before slot i = min(sum of the earlier slots' wishes, B)   (a saturating sum of non-negative terms)
// so every lane derives exactly the values the sequential loop would have reached at its slot; the result is identical
// entry for entry (checked against the C restatement after every iteration by the GPU scheduler tests).
// Each lane's dependent loads (request id -> step -> token row) then overlap with the other lanes', which is what the
// sequential version spends its time on (about 1.8 us per occupied slot).  `lds` holds the page-table snapshot
// ([0, NP)) and the pages retired in this step in ring order ([NP, 2 NP)): a page returned by one lane and handed out
// again by another in the same step goes through LDS, never through a store and a load of different lanes.
__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __builtin_amdgcn_ds_bpermute(((lane - o) & 63) << 2, v);
    if (lane >= o) v += u;
  }
  return v;
}
__device__ __forceinline__ int wave_bcast(int v, int src) { return __builtin_amdgcn_readlane(v, src); }

// `portion` > 0: one that runs beside those just prepared, in the same iteration (MK_PAIR_NEXT in the result of the step that prepared the last of them).
#define MK_PAIR_NEXT (1 << 16)
__device__ __attribute__((noinline)) int mk_prepare_next_batch_wave(const MkRuntime &rt, int *lds, int lane, int portion) {
  const int second = MK_PAIR ? portion * MK_MAX_TOKENS : 0;
  long long *const ids = second ? rt.ids2 + second - MK_MAX_TOKENS : rt.input_tokens;
  MkSched *sc = rt.sched;
  const int R = rt.max_requests, B = rt.max_tokens, PS = rt.page_size, NP = rt.max_pages;
  int *snap = lds, *freed = lds + NP;
  const int head0 = sc->page_queue_head, tail0 = sc->page_queue_tail;
  const int old_pages = rt.kv_indptr[R];
  // 1. commit the previous iteration's outputs, find the requests that retire
  const bool slot = lane < R;
  int req = slot ? rt.request_ids[lane] : -1;
  int st = 0, plen = 0, k0 = 0, k1 = 0;
  bool retire = false;
  if (req >= 0) {
    st = rt.step[req];
    const int q0 = rt.qo_indptr[lane];
    const int n = rt.qo_indptr[lane + 1] - q0;
    plen = rt.prompt_lengths[req];
    k0 = rt.kv_indptr[lane];
    k1 = rt.kv_indptr[lane + 1];
    for (int j = 0; j < n; j++) {
      const int pos = st + j + 1;
      if (pos >= plen && pos < rt.max_seq) rt.tokens[(long long)req * rt.max_seq + pos] = rt.output_tokens[q0 + j];
    }
    st += n;
    rt.step[req] = st;
    const bool full = st + 1 >= rt.max_seq;
    const bool eos = st >= plen && rt.tokens[(long long)req * rt.max_seq + st] == rt.eos_token_id;
    retire = full || eos;
  }
  // 2. snapshot the page table; retired pages go back to the ring in slot order
  for (int i = lane; i < old_pages; i += 64) snap[i] = rt.kv_indices[i];
  const int rp = retire ? k1 - k0 : 0;
  const int rp_incl = wave_incl_scan(rp, lane);
  const int n_freed = wave_bcast(rp_incl, 63);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  for (int j = 0; j < rp; j++) {
    const int pg = snap[k0 + j], at = rp_incl - rp + j;
    freed[at] = pg;
    rt.page_queue[(tail0 + at) % NP] = pg;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  const int avail0 = tail0 - head0;  // pages the ring held before this step
  auto ring_page = [&](int a) -> int {  // the a-th page handed out in this step
    return a < avail0 ? rt.page_queue[(head0 + a) % NP] : freed[a - avail0];
  };
  // 3. running requests keep their slot order, compacted over retired slots
  const bool alive = req >= 0 && !retire;
  const unsigned long long alive_mask = __ballot(alive);
  const int rank = __popcll(alive_mask & ((1ull << lane) - 1ull));
  const int nrun = __popcll(alive_mask);
  if (rt.state_ids && slot) {  // recurrent-state slots: the survivors' in front, in order, then the free ones
    const int id = rt.state_ids[lane];
    rt.state_ids[alive ? rank : nrun + (lane - rank)] = id;
  }
  const int wish = alive ? (plen - st > 0 ? min(plen - st, rt.max_new_per_req) : 1) : 0;
  const int wish_incl = wave_incl_scan(wish, lane);
  const int tok0 = min(wish_incl - wish, B), n = min(wish_incl, B) - tok0;
  const int had = alive ? k1 - k0 : 0;
  const int need = alive ? (st + n + PS - 1) / PS : 0;
  const int need_incl = wave_incl_scan(need, lane);
  const int fresh = need > had ? need - had : 0;
  const int fresh_incl = wave_incl_scan(fresh, lane);
  if (alive) {
    const int page0 = need_incl - need, a0 = fresh_incl - fresh;
    rt.request_ids[rank] = req;
    rt.qo_indptr[rank] = tok0;
    rt.kv_indptr[rank] = page0;
    const int last = (st + n) % PS;
    rt.kv_last_page_len[rank] = last == 0 ? PS : last;
    for (int j = 0; j < had && j < need; j++) rt.kv_indices[page0 + j] = snap[k0 + j];
    for (int j = had; j < need; j++) rt.kv_indices[page0 + j] = ring_page(a0 + j - had);
  }
  // Rows of the slots' lanes, [t0, t0 + n) of request q from position p on: a slot's own lane writes them one after the other, or, where that
  // takes more turns than there are slots with several, all lanes write one slot's rows after the other's (a portion of 64 tokens of one
  // request behind 2432: 29.4 us a step by the sequential one, 12.9 by this; of 9, 16 and 32 tokens behind forty such 8.7 / 7.7, 10.8 / 8.6, 17.0 / 10.0).
  auto rows = [&](int n, int t0, int q, int p, int at) {
    int most = 0;
#pragma unroll
    for (int b = 64; b; b >>= 1)
      if (__any(n >= most + b)) most += b;
    auto write = [&](int row, int first, int rq, int pos, int slot_) {
      ids[row] = rt.tokens[(long long)rq * rt.max_seq + pos];
      rt.tok_slot[row + second] = slot_;
      rt.tok_pos[row + second] = pos;
      rt.tok_first[row + second] = first;
    };
    unsigned long long several = __ballot(n > 1);
    const bool shared = __popcll(several) < most;
    for (int j = 0; j < (shared && n > 1 ? 0 : n); j++) write(t0 + j, t0, q, p + j, at);
    while (shared && several) {
      const int l = (int)__ffsll(several) - 1;
      several &= several - 1;
      const int t_ = wave_bcast(t0, l), q_ = wave_bcast(q, l), p_ = wave_bcast(p, l), at_ = wave_bcast(at, l);
      if (lane < wave_bcast(n, l)) write(t_ + lane, t_, q_, p_ + lane, at_);
    }
  };
  rows(n, tok0, req, st, rank);
  int ntok = min(wave_bcast(wish_incl, 63), B);
  int npage = wave_bcast(need_incl, 63);
  int taken = wave_bcast(fresh_incl, 63);
  int nreq = nrun;
  bool inner = rt.max_new_per_req > 1 && !__any(n > 0 && (st + n >= plen || st + n + 1 >= rt.max_seq));
  bool pairs = false;  // the next portion could run in the same iteration: nothing hangs on this one's samples, it is full, and lies inside prompts
  // 4. admit new requests while there is room: lane k looks at request next_request_id + k
  {
    const int next = sc->next_request_id;
    const int cand = next + lane;
    const bool valid = nreq + lane < R && cand < rt.total_requests;
    const int cplen = valid ? rt.prompt_lengths[cand] : 0;
    const int cwish = valid ? min(cplen, rt.max_new_per_req) : 0;
    const int cw_incl = wave_incl_scan(cwish, lane);
    // the sequential loop reaches candidate k only while the budget is not exhausted, and stops at the first request
    // that does not exist; candidates are valid in a prefix of the lanes, so "admitted" is a prefix too
    const bool admit = valid && ntok + (cw_incl - cwish) < B;
    const int cn = admit ? min(cwish, B - (ntok + cw_incl - cwish)) : 0;
    const int cneed = admit ? (cn + PS - 1) / PS : 0;
    const int cneed_incl = wave_incl_scan(cneed, lane);
    const int n_admit = __popcll(__ballot(admit));
    inner = inner && !__any(admit && (cn >= cplen || cn + 1 >= rt.max_seq));
    if (admit) {
      const int s_ = nreq + lane, tok0c = ntok + cw_incl - cwish, page0 = npage + cneed_incl - cneed, a0 = taken + cneed_incl - cneed;
      rt.request_ids[s_] = cand;
      rt.qo_indptr[s_] = tok0c;
      rt.kv_indptr[s_] = page0;
      const int last = cn % PS;
      rt.kv_last_page_len[s_] = last == 0 ? PS : last;
      for (int j = 0; j < cneed; j++) rt.kv_indices[page0 + j] = ring_page(a0 + j);
    }
    rows(cn, ntok + cw_incl - cwish, cand, 0, nreq + lane);
    if (MK_PAIR && rt.pair_n) {
      const int w1 = alive ? min(plen - st - n, rt.max_new_per_req) : 0, i1 = wave_incl_scan(w1, lane), s1 = wave_bcast(i1, 63);
      const int w2 = admit ? min(cplen - cn, rt.max_new_per_req) : 0, i2 = s1 + wave_incl_scan(w2, lane);
      const int n1 = min(i1, B) - min(i1 - w1, B), n2 = min(i2, B) - min(i2 - w2, B);
      const bool ends = (n1 > 0 && (st + n + n1 >= plen || st + n + n1 + 1 >= rt.max_seq)) || (n2 > 0 && (cn + n2 >= cplen || cn + n2 + 1 >= rt.max_seq));
      pairs = inner && wave_bcast(i2, 63) >= B && !__any(ends);
    }
    const int cn_incl = wave_incl_scan(cn, lane);
    ntok += wave_bcast(cn_incl, 63);
    npage += wave_bcast(cneed_incl, 63);
    taken += wave_bcast(cneed_incl, 63);
    nreq += n_admit;
    if (lane == 0) sc->next_request_id = next + n_admit;
  }
  // 5. clear unused slots
  for (int i = nreq + lane; i < R; i += 64) rt.request_ids[i] = -1;
  for (int i = nreq + lane; i <= R; i += 64) {
    rt.qo_indptr[i] = ntok;
    rt.kv_indptr[i] = npage;
  }
  if (lane == 0) {
    sc->page_queue_head = head0 + taken;
    sc->page_queue_tail = tail0 + n_freed;
    if (MK_PAIR) sc->group[portion] = ntok;
    if (!second) {
      sc->num_tokens = ntok;
      sc->inner = inner;
    }
    sc->num_reqs = nreq;
  }
  return pairs && 2 * ntok > B ? ntok | MK_PAIR_NEXT : ntok;
}

// Batch description for a launch whose batch the HOST prepared (the reference's MODE_ONLINE_NOTOKEN, one pass per launch,
// persistent_kernel.cuh:570-582, and MODE_ONEPASS): the caller has filled input_tokens, qo_indptr, paged_kv_indptr,
// paged_kv_indices and paged_kv_last_page_len the way the reference's attention tasks read them -- request slot i owns
// rows [qo_indptr[i], qo_indptr[i+1]) and its sequence, new tokens included, is (pages - 1) * page_size + last_page_len
// long, so its rows sit at the last positions of that sequence.  Derives the per-row slot / position / first-row arrays
// on the device (no host round trip, so a serving loop can enqueue launches back to back).
// Runs on a wavefront, a lane per batch slot, so that the slots' loads overlap (one thread took one to two microseconds per slot).  Reads and
// writes at device scope: mk_fetch_batch may have written the tensors a moment ago, and nobody releases behind the step.
// `off`: words to the description of a portion that runs beside the first one in the same iteration (0: the first one's); what is looked up by
// slot lies there as well.  `several`: there are such portions, this one being the `portion`-th.
__device__ __forceinline__ int mk_batch_from_meta(const MkRuntime &rt, int lane, int off, bool several, int portion) {
  const int R = rt.max_requests, B = rt.max_tokens, second = MK_PAIR ? portion * MK_MAX_TOKENS : 0;
  // A batch the stages cannot run as described is not run at all: truncating a request's rows would leave the rest with
  // the slot / position an earlier launch gave them, and they would append K/V rows to some other request's cache.
  // bad, of the first slot that cannot run: 1 = rows outside [0, max tokens), overlapping, or with gaps; 2 = more rows for one
  // request than max_tokens_per_request; 3 = a sequence shorter than its new rows, longer than max_seq_length, or without pages.
  const int i = min(lane, R - 1);  // (at most 64 slots)
  const int q0 = ldc_i32(rt.qo_indptr + off + i), q1 = ldc_i32(rt.qo_indptr + off + i + 1), pages = ldc_i32(rt.kv_indptr + off + i + 1) - ldc_i32(rt.kv_indptr + off + i),
            last = ldc_i32(rt.kv_last_page_len + off + i);
  const int n = lane < R ? q1 - q0 : 0;  // (<= 0: an unused slot; hosts that fill only the first entries leave zeros behind them)
  const int len = (int)((long long)(pages - 1) * rt.page_size) + last;
  const bool inside = n > 0 && q0 >= 0 && n <= B && q0 <= B - n;
  const unsigned long long rows = inside ? (n >= 64 ? ~0ull : ((1ull << n) - 1ull)) << q0 : 0ull;
  unsigned lo = (unsigned)rows, hi = (unsigned)(rows >> 32);  // rows of this slot and those in front of it
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned ul = (unsigned)__builtin_amdgcn_ds_bpermute(((lane - o) & 63) << 2, (int)lo), uh = (unsigned)__builtin_amdgcn_ds_bpermute(((lane - o) & 63) << 2, (int)hi);
    if (lane >= o) {
      lo |= ul;
      hi |= uh;
    }
  }
  const unsigned pl = (unsigned)__builtin_amdgcn_ds_bpermute(((lane - 1) & 63) << 2, (int)lo), ph = (unsigned)__builtin_amdgcn_ds_bpermute(((lane - 1) & 63) << 2, (int)hi);
  const unsigned long long before = lane ? (unsigned long long)pl | ((unsigned long long)ph << 32) : 0ull;
  const int why = n <= 0 ? 0 : !inside ? 1 : n > rt.max_new_per_req ? 2 : (before & rows) ? 1 : pages < 1 || len < n || len > rt.max_seq ? 3 : 0;
  const unsigned long long which = __ballot(why != 0);
  int bad = which ? wave_bcast(why, (int)__ffsll(which) - 1) : 0;
  const unsigned long long covered = (unsigned long long)(unsigned)wave_bcast((int)lo, 63) | ((unsigned long long)(unsigned)wave_bcast((int)hi, 63) << 32);
  int ntok = covered ? 64 - __clzll((long long)covered) : 0;
  if (covered != (ntok >= 64 ? ~0ull : ((1ull << ntok) - 1ull)) && !bad) bad = 1;
  if (several && ntok < 3 && !bad) bad = 4;
  if (bad) ntok = 0;
  // a lane per row (by the lanes of the slots, row after row, 64 rows of one request took 16 us)
  int slot = 0, first = 0, pos = 0;
  for (unsigned long long live = ntok ? __ballot(n > 0) : 0ull; live; live &= live - 1) {
    const int s = (int)__ffsll(live) - 1, f = wave_bcast(q0, s);
    if (lane >= f && lane < wave_bcast(q1, s)) {
      slot = s;
      first = f;
      pos = wave_bcast(len, s) - wave_bcast(q1, s) + lane;
    }
  }
  if (lane < ntok) {
    stc_i32(rt.tok_slot + second + lane, off + slot);
    stc_i32(rt.tok_pos + second + lane, pos);
    stc_i32(rt.tok_first + second + lane, first);
    if (second) stc_u64(rt.ids2 + second - MK_MAX_TOKENS + lane, ldc_u64((const int *)rt.input_tokens + off + 2 * lane));
  }
  const bool single = !__any(n > 1);
  if (lane == 0) {
    if (several) {  // (where one is bad, none of them runs: mk_kernel_body)
      stc_i32(&rt.sched->group[portion], bad ? -bad : single ? ntok | MK_GROUP_SINGLE : ntok);
    } else {
      stc_i32(&rt.sched->bad_batch, bad);
      stc_i32(&rt.sched->num_tokens, ntok);
    }
  }
  return ntok;
}

// The words of a batch in pinned host memory go where the stages read them, by one wavefront, each word read once.  Bound by one round trip
// over the bus, 2 us for up to 2048 words.  (As a copy on the stream in front of the launch it cost 12: a cooperative
// launch sits on a queue of its own and waits for the copy's signal.  Words behind the end read again as the first ones, as elsewhere here, made it
// 18 to 40: lines that the host has just written are slow to fetch, every time.)
__device__ __forceinline__ void mk_fetch_batch(const int *src, int *dst, long long words, int lane) {
  for (long long i = lane; i < words; i += 32 * 64) {
    int v[32];
#pragma unroll
    for (int k = 0; k < 32; k++)
      if (i + k * 64 < words) v[k] = __hip_atomic_load(src + i + k * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
#pragma unroll
    for (int k = 0; k < 32; k++)
      if (i + k * 64 < words) stc_i32(dst + i + k * 64, v[k]);
  }
}

// The scheduler's step of a launch whose batch the host describes, by one wavefront of the first workgroup, beside the handshake that opens the
// launch: behind it, on the first virtual workgroup, its 5.6 us came on top (13 passes of suborax-small 2005 -> 1980 us).
__device__ __attribute__((noinline)) void mk_open_batch(const MkRuntime &rt, int lane, const int *src, int *dst, long long words) {
  if (words) mk_fetch_batch(src, dst, words, lane);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  const int ntok = mk_batch_from_meta(rt, lane, 0, false, 0);
  if (lane == 0) {
    MkSched *sc = rt.sched;
    if (ntok == 0) sc->finished = 1;
    else sc->iterations += 1;
    if (rt.timing && sc->iterations <= rt.timing_cap) rt.timing[sc->iterations] = (long long)wall_clock64();
  }
}
#if MK_PAIR
// The same for one portion of several, each by a workgroup of its own (one after the other, a portion takes 4 to 6 us); what the launch makes of them
// all is for mk_kernel_body.
__device__ __attribute__((noinline)) void mk_open_portion(const MkRuntime &rt, int lane, const int *src, int *dst, int words, int off, int portion, int portions) {
  if (words) mk_fetch_batch(src + off, dst + off, words, lane);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  mk_batch_from_meta(rt, lane, off, true, portion);
  if (lane == 0 && portion == portions - 1 && portions < MK_GROUP) stc_i32(&rt.sched->group[portions], 0);
}
#endif

// The reference's MODE_ONLINE step (persistent_kernel.cuh:538-568): one request (slot 0, request 0) whose tokens the
// host has written into tokens[0, :]; every pass consumes num_new_tokens[0] of them starting at step[0].  After a pass
// step[0] advances by what the pass consumed, and the run ends when the position it started from is within two of
// max_seq_length or the token after it is the EOS id -- the reference's test, on the step value from before the
// advance.  What the reference leaves to the host and is done here instead: the page table of the one request
// (identity: page j of the ring is page j of the sequence) and the qo / kv index arrays.  Runs on one thread.
__device__ __attribute__((noinline)) int mk_online_next_batch(const MkRuntime &rt) {
  MkSched *sc = rt.sched;
  const int PS = rt.page_size;
  int step = rt.step[0];
  if (sc->online_started) {
    const int consumed = sc->num_tokens;
    rt.step[0] = step + consumed;
    const bool stop = (step + 2 >= rt.max_seq) || (rt.tokens[step + 1] == rt.eos_token_id);
    step += consumed;
    if (stop) {
      sc->num_tokens = 0;
      return 0;
    }
  }
  sc->online_started = 1;
  int n = rt.num_new_tokens ? rt.num_new_tokens[0] : 1;
  n = n < 1 ? 1 : n;
  n = min(n, min(rt.max_new_per_req, rt.max_tokens));
  n = min(n, rt.max_seq - 1 - step);
  if (n <= 0) {
    sc->num_tokens = 0;
    return 0;
  }
  for (int j = 0; j < n; j++) {
    rt.input_tokens[j] = rt.tokens[step + j];
    rt.tok_slot[j] = 0;
    rt.tok_pos[j] = step + j;
    rt.tok_first[j] = 0;
  }
  const int need = (step + n + PS - 1) / PS, last = (step + n) % PS;
  rt.request_ids[0] = 0;
  rt.kv_last_page_len[0] = last == 0 ? PS : last;
  for (int j = 0; j < need && j < rt.max_pages; j++) rt.kv_indices[j] = j;
  rt.qo_indptr[0] = 0;
  rt.kv_indptr[0] = 0;
  for (int i = 1; i <= rt.max_requests; i++) {
    rt.qo_indptr[i] = n;
    rt.kv_indptr[i] = need;
  }
  sc->num_tokens = n;
  sc->num_reqs = 1;
  return n;
}

// ----------------------------------------------------------------------------- weights
__device__ __forceinline__ const u32x4 *weight_row(CWeight &w, int r, int k8) {
  if (w.nseg == 1) return (const u32x4 *)w.seg[0] + (size_t)r * k8;
  const int g = r / w.group_rows;
  int o = r - g * w.group_rows;
  int s = 0;
  if (o >= w.seg_rows[0]) {
    o -= w.seg_rows[0];
    s = 1;
    if (w.nseg > 2 && o >= w.seg_rows[1]) {
      o -= w.seg_rows[1];
      s = 2;
    }
  }
  return (const u32x4 *)w.seg[s] + (size_t)(g * w.seg_rows[s] + o) * k8;
}

// ----------------------------------------------------------------------------- stages
// Every stage function posts barrier_wait(c) itself, after any work that does not depend on the previous
// stage (weight prefetch), and the main loop posts barrier_arrive(c) when the function returns.

// The row a workgroup takes first where rows are dealt round-robin over the dies (and then every G-th).  A second portion's rows, in a stage that has
// just dealt the first one's, go to the workgroups behind those.
__device__ __forceinline__ int row_item(const Ctx &c, int t) {
#if MK_PAIR
  return mk_first_row(t, c.rows_ahead, c.G);
#else
  return t;
#endif
}
__device__ __forceinline__ int row_item(const Ctx &c) { return row_item(c, c.even_xcds ? c.rank * c.nxcd + c.xi : c.vid); }

// Gather embedding rows.  Reference task: tasks/ampere/embedding.cuh:42-72.
__device__ __forceinline__ void stage_embed(CStage &st, Ctx &c, const MkRuntime &rt, int M) {
  barrier_wait(c);
  const int k8 = st.k / 8;
  for (int t = row_item(c, c.vid); t < M; t += c.G) {
    long long id;
    if (st.flags & MK_F_EMBED_FROM_TOKENS) {
      const int req = ldc_i32(&rt.request_ids[c.sh_tok[MK_MAX_TOKENS + t]]);
      id = (long long)ldc_u64(&rt.tokens[(long long)req * rt.max_seq + c.sh_tok[t]]);
    } else {
      id = (long long)ldc_u64((const long long *)st.in + t);
    }
    const u32x4 *src = (const u32x4 *)st.w.seg[0] + (size_t)(id < 0 ? 0 : id) * k8;
    u32x4 *dst = (u32x4 *)st.out + (size_t)t * (st.ld_out / 8);
    const u32x4 zero = {0u, 0u, 0u, 0u};
    for (int i = c.tid; i < k8; i += MK_THREADS) dst[i] = id < 0 ? zero : src[i];
  }
}

// Block-wide sum of one float per thread.
__device__ __forceinline__ float block_sum(float v, float *red) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

// RMSNorm of full rows, one workgroup per token row (used when an iteration has several tokens;
// single-token iterations fuse the norm into the consuming linear).  y = bf16((x * r) * w) with
// r = rsqrt(mean(x^2) + eps) in fp32.  Reference task: tasks/mi300/rmsnorm_mi300.cuh:37-188.
//
// NS 16-byte segments per thread: the norm weights are requested before the barrier is awaited, the row is read with device-scope
// loads and written through, so the arrival needs no L2 write-back.  Bound by the barrier and one round trip for the row, so everything
// a row needs (of up to 512 segments with up to four slices: every slice of every segment) is requested before the first value is
// waited for; a branch around each segment had made a round trip per segment of it.
// 4096 values from four slices, as a stage: 8.4 -> 7.3 us, now 5.4.
template <int NS>
__device__ __forceinline__ void stage_norm_rows(CStage &st, Ctx &c, int M, char *smem) {
  const int tid = c.tid, k8 = st.k / 8;
  float *red = (float *)smem;
  const u32x4 *w4 = (const u32x4 *)st.norm_w;
  auto at = [&](int j) { return min(tid + j * MK_THREADS, k8 - 1); };
  auto on = [&](int j) { return NS <= 2 || j * MK_THREADS < k8; };  // (long rows: segments nobody has are left out)
  u32x4 g[NS], v[NS];
#pragma unroll
  for (int j = 0; j < NS; j++)
    if (on(j)) g[j] = w4[at(j)];
  barrier_wait(c);
  const int dS = c.defer_S;
  c.defer_S = 0;
  // rows are dealt round-robin over the dies, so a handful of rows does not funnel through one die's memory path
  const int t0 = row_item(c);
  for (int t = t0; t < M; t += c.G) {
    const u32x4 *x = (const u32x4 *)((const uint16_t *)st.in + (size_t)t * st.ld_in);
    u32x4 *y = (u32x4 *)((uint16_t *)st.out + (size_t)t * st.ld_out);
    float ss = 0.f;
    if (dS) {
      // the rows are still K-slice partials: finish the producing linear (sum in slice order, residual, rounding), store its output
      // row where it belongs, and normalise the rounded values
      const u32x4 *r4 = (const u32x4 *)((const uint16_t *)c.defer_res + (size_t)t * c.defer_ld_res);
      auto sum_slices = [&](auto ns) {
        constexpr int Q = decltype(ns)::value, JB = NS * Q <= 8 ? NS : 1;  // segments requested together
#pragma unroll
        for (int j0 = 0; j0 < NS; j0 += JB) {
          if (!on(j0)) continue;
          u32x4 pv[JB][Q][2], rv[JB];
          __amdgpu_buffer_rsrc_t rows[Q];
#pragma unroll
          for (int q = 0; q < Q; q++) rows[q] = dev_rows(c.defer_part + ((size_t)q * c.defer_rows + t) * st.k);
#pragma unroll
          for (int j = 0; j < JB; j++) {
            const int seg = at(j0 + j);
            rv[j] = ldc_16B(c.defer_res ? r4 + seg : (const u32x4 *)c.defer_part);
#pragma unroll
            for (int q = 0; q < Q; q++) {
              pv[j][q][0] = ldc_16B(rows[q], seg * 32);
              pv[j][q][1] = ldc_16B(rows[q], seg * 32 + 16);
            }
          }
#pragma unroll
          for (int j = 0; j < JB; j++) {
            float a[8];
#pragma unroll
            for (int e = 0; e < 8; e++) a[e] = 0.f;
#pragma unroll
            for (int q = 0; q < Q; q++)
#pragma unroll
              for (int e = 0; e < 4; e++) {
                a[e] += __uint_as_float(pv[j][q][0][e]);
                a[4 + e] += __uint_as_float(pv[j][q][1][e]);
              }
            if (c.defer_res) {
#pragma unroll
              for (int e = 0; e < 4; e++) {
                a[2 * e] += bf_lo(rv[j][e]);
                a[2 * e + 1] += bf_hi(rv[j][e]);
              }
            }
#pragma unroll
            for (int e = 0; e < 4; e++) v[j0 + j][e] = pack2(a[2 * e], a[2 * e + 1]);
          }
        }
      };
      if (dS == 2) sum_slices(std::integral_constant<int, 2>{});
      else if (dS == 4) sum_slices(std::integral_constant<int, 4>{});
      else sum_slices(std::integral_constant<int, 8>{});
#pragma unroll
      for (int j = 0; j < NS; j++)  // stores after all the loads: neither is moved across the other
        if (tid + j * MK_THREADS < k8) stc_16B((u32x4 *)x + tid + j * MK_THREADS, v[j]);
    } else {
#pragma unroll
      for (int j = 0; j < NS; j++)
        if (on(j)) v[j] = ldc_16B(x + at(j));
    }
#pragma unroll
    for (int j = 0; j < NS; j++) {
      if (!on(j)) continue;
      const bool ok = tid + j * MK_THREADS < k8;
#pragma unroll
      for (int e = 0; e < 4; e++) ss += ok ? bf_lo(v[j][e]) * bf_lo(v[j][e]) + bf_hi(v[j][e]) * bf_hi(v[j][e]) : 0.f;
    }
    ss = block_sum(ss, red);
    const float r = rsqrtf(ss / (float)st.k + st.eps);
#pragma unroll
    for (int j = 0; j < NS; j++)
      if (tid + j * MK_THREADS < k8) {
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = pack2((bf_lo(v[j][e]) * r) * bf_lo(g[j][e]), (bf_hi(v[j][e]) * r) * bf_hi(g[j][e]));
        stc_16B(y + tid + j * MK_THREADS, o);
      }
    __syncthreads();
  }
  c.wrote_through = true;
}
__device__ __forceinline__ void stage_norm(CStage &st, Ctx &c, int M, char *smem) {
  const int k8 = st.k / 8;
  if (mk_norm_by_rows(st)) {
    if (k8 <= MK_THREADS) stage_norm_rows<1>(st, c, M, smem);
    else if (k8 <= 2 * MK_THREADS) stage_norm_rows<2>(st, c, M, smem);
    else stage_norm_rows<6>(st, c, M, smem);
    return;
  }
  barrier_wait(c);
  float *red = (float *)smem;
  uint32_t *xs = (uint32_t *)(smem + 1024);
  const int k2 = st.k / 2;
  for (int t = c.vid; t < M; t += c.G) {
    const uint32_t *x = (const uint32_t *)st.in + (size_t)t * (st.ld_in / 2);
    const uint32_t *w = (const uint32_t *)st.norm_w;
    uint32_t *y = (uint32_t *)st.out + (size_t)t * (st.ld_out / 2);
    float ss = 0.f;
    for (int i = c.tid; i < k2; i += MK_THREADS) {
      const uint32_t u = ldc_u32(x + i);
      xs[i] = u;
      ss += bf_lo(u) * bf_lo(u) + bf_hi(u) * bf_hi(u);
    }
    ss = block_sum(ss, red);
    const float r = rsqrtf(ss / (float)st.k + st.eps);
    for (int i = c.tid; i < k2; i += MK_THREADS) {
      const uint32_t u = xs[i], g = w[i];
      y[i] = pack2((bf_lo(u) * r) * bf_lo(g), (bf_hi(u) * r) * bf_hi(g));
    }
    __syncthreads();
  }
}

__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.f + __expf(-g)) * u; }
// gated activation of a [gate ; up] linear (dual kernels: gelu where the stage asks for it, 32-bit: library functions)
__device__ __forceinline__ float gelu_tanh(float z) {  // z / (1 + e^-2y) = z (1 + tanh y) / 2
  return z / (1.f + __expf(-1.5957691216057308f * (z + 0.044715f * z * z * z)));
}
__device__ __forceinline__ float linear_glu(CStage &st, float g, float u) {
#if MK_HAVE_DUAL
  if (st.flags & MK_F_GELU) return gelu_tanh(g) * u;
#endif
  return silu_mul(g, u);
}
// activation of a plain linear's outputs (hybrid kernels: the square of relu where the stage asks for it)
__device__ __forceinline__ float linear_act(CStage &st, float v) {
#if MK_HAVE_HYB
  const float p = fmaxf(v, 0.f);
  return (st.flags & MK_F_RELU2) ? p * p : v;
#else
  return v;
#endif
}

#if MK_HAVE_MIX  // a residual_prenorm in front of a single-token linear (mk_mix.hip): by the workgroup, by the control wavefront
__device__ __forceinline__ void mx_x_m1_prenorm(CStage &st, const Ctx &c, uint32_t *xs, float *red);
template <int KL> __device__ __forceinline__ void mx_x_m1_prenorm_wave(CStage &st, Ctx &c, uint32_t *xs, int lane);
__device__ __forceinline__ bool mx_linear_m1_form(CStage &st);
__device__ __forceinline__ void stage_mx_linear_m1(CStage &st, Ctx &c, char *smem);
// the control wavefront wants whole 16-byte segments in one part of the norm, and few parts
__device__ __forceinline__ bool mx_prenorm_by_wave(CStage &st) { return st.k <= 4096 && st.norm_groups <= 8 && (st.k_real / st.norm_groups & 7) == 0; }
#endif

// Stage the single input row of a one-token linear in LDS as packed bf16, applying the fused RMSNorm when the
// stage asks for it (virtual workgroup 0 also stores the normalised row, which is the norm task's output tensor).
// FX: the norm in front may be an FX_ADDNORM (see mk_flex.hip): alpha * residual + y, both rows in memory, then the norm.
template <bool FX>
__device__ __forceinline__ void stage_x_m1(CStage &st, const Ctx &c, uint32_t *xs, float *red) {
  const int tid = c.tid, k4 = st.k / 4;
  const unsigned long long *xin = (const unsigned long long *)st.in;
  unsigned long long *xs2 = (unsigned long long *)xs;
  if constexpr (FX) {
#if MK_HAVE_MIX
    if (st.flags & MK_F_PRENORM) {
      mx_x_m1_prenorm(st, c, xs, red);
      return;
    }
#endif
    if (st.flags & MK_F_ADDNORM) {
      f32x4 *vs = (f32x4 *)((char *)xs + MK_MOE_OFFSET);  // the sum, 32-bit
      float ss = 0.f;
      for (int i = tid; i < k4; i += MK_THREADS) {
        const f32x4 x = __builtin_bit_cast(f32x4, ldc_16B((const u32x4 *)st.res + i));
        const unsigned long long u = st.y_in ? ldc_u64((const unsigned long long *)st.y_in + i) : 0ull;
        const uint32_t a = (uint32_t)u, b = (uint32_t)(u >> 32);
        const f32x4 v = {fmaf(st.alpha, x[0], bf_lo(a)), fmaf(st.alpha, x[1], bf_hi(a)), fmaf(st.alpha, x[2], bf_lo(b)), fmaf(st.alpha, x[3], bf_hi(b))};
        vs[i] = v;
        ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
      }
      ss = block_sum(ss, red);
      const float r = 1.f / sqrtf(ss / (float)st.k_real + st.norm_eps);
      for (int i = tid; i < k4; i += MK_THREADS) {
        const f32x4 g = ((const f32x4 *)st.norm_w)[i], v = vs[i];
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (v[e] * r) * (st.w_offset + g[e]);
        const unsigned long long h = (unsigned long long)pack2(o[0], o[1]) | ((unsigned long long)pack2(o[2], o[3]) << 32);
        xs2[i] = h;
        if (c.vid == 0) {
          if (st.out2) stc_16B((u32x4 *)st.out2 + i, __builtin_bit_cast(u32x4, o));
          stc_u64((unsigned long long *)st.norm_out + i, h);
        }
      }
      __syncthreads();
      return;
    }
  }
  if (st.flags & MK_F_NORM) {
    float ss = 0.f;
    for (int i = tid; i < k4; i += MK_THREADS) {
      const unsigned long long u = ldc_u64(xin + i);
      xs2[i] = u;
      const uint32_t a = (uint32_t)u, b = (uint32_t)(u >> 32);
      ss += bf_lo(a) * bf_lo(a) + bf_hi(a) * bf_hi(a) + bf_lo(b) * bf_lo(b) + bf_hi(b) * bf_hi(b);
    }
    ss = block_sum(ss, red);
    const float r = rsqrtf(ss / (float)st.k + st.eps);
    const uint32_t *nw = (const uint32_t *)st.norm_w;
    uint32_t *no = (c.vid == 0) ? (uint32_t *)st.norm_out : nullptr;
    for (int i = tid; i < st.k / 2; i += MK_THREADS) {
      const uint32_t u = xs[i], g = nw[i];
      const uint32_t y = pack2((bf_lo(u) * r) * bf_lo(g), (bf_hi(u) * r) * bf_hi(g));
      xs[i] = y;
      if (no) no[i] = y;
    }
  } else {
    for (int i = tid; i < k4; i += MK_THREADS) xs2[i] = ldc_u64(xin + i);
  }
  __syncthreads();
}

// Same staging done by ONE wavefront (the control wavefront of a tuned single-token linear): lane l owns the
// 16-byte segments l, l+64, ... of the row, the sum of squares is a wavefront reduction, no workgroup barrier inside.
template <int KL>
__device__ __forceinline__ void stage_x_m1_wave(CStage &st, const Ctx &c, uint32_t *xs, int lane, const u32x4 (&nwv)[KL]) {
  const u32x4 *xin = (const u32x4 *)st.in;
  u32x4 *xs4 = (u32x4 *)xs;
  u32x4 v[KL];
#pragma unroll
  for (int kc = 0; kc < KL; kc++) v[kc] = ldc_16B(xin + kc * 64 + lane);
  if (st.flags & MK_F_NORM) {
    float ss = 0.f;
#pragma unroll
    for (int kc = 0; kc < KL; kc++) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t u = v[kc][e];
        ss += bf_lo(u) * bf_lo(u) + bf_hi(u) * bf_hi(u);
      }
    }
    ss = wave_sum(ss);
    const float r = rsqrtf(ss / (float)(KL * 512) + st.eps);
    u32x4 *no = (c.vid == 0) ? (u32x4 *)st.norm_out : nullptr;
#pragma unroll
    for (int kc = 0; kc < KL; kc++) {
      const u32x4 g = nwv[kc];  // norm weights were requested before the barrier was awaited
      u32x4 y;
#pragma unroll
      for (int e = 0; e < 4; e++) y[e] = pack2((bf_lo(v[kc][e]) * r) * bf_lo(g[e]), (bf_hi(v[kc][e]) * r) * bf_hi(g[e]));
      xs4[kc * 64 + lane] = y;
      if (no) stc_16B(no + kc * 64 + lane, y);
    }
  } else {
#pragma unroll
    for (int kc = 0; kc < KL; kc++) xs4[kc * 64 + lane] = v[kc];
  }
}

// ... with an FX_ADDNORM in front: the norm weights and, where the previous stage does not write them, the residual values
// were requested before the barrier was awaited.
template <int KL>
__device__ __forceinline__ void stage_x_m1_addnorm_wave(CStage &st, Ctx &c, uint32_t *xs, int lane) {
  const f32x4 *w4 = (const f32x4 *)st.norm_w;
  const u32x4 *x4 = (const u32x4 *)st.res;
  f32x4 g[KL][2], x[KL][2];
  auto load_x = [&]() {
#pragma unroll
    for (int kc = 0; kc < KL; kc++)
#pragma unroll
      for (int h = 0; h < 2; h++) x[kc][h] = __builtin_bit_cast(f32x4, ldc_16B(x4 + (kc * 64 + lane) * 2 + h));
  };
#pragma unroll
  for (int kc = 0; kc < KL; kc++)
#pragma unroll
    for (int h = 0; h < 2; h++) g[kc][h] = w4[(kc * 64 + lane) * 2 + h];
  const bool early = st.flags & MK_F_RES_EARLY;
  if (early) load_x();
  if (c.pending && lane == 0) barrier_poll(c);
  if (!early) load_x();
  u32x4 y[KL];
#pragma unroll
  for (int kc = 0; kc < KL; kc++) y[kc] = st.y_in ? ldc_16B((const u32x4 *)st.y_in + kc * 64 + lane) : (u32x4){0u, 0u, 0u, 0u};
  float ss = 0.f;
#pragma unroll
  for (int kc = 0; kc < KL; kc++)
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t u = y[kc][h * 2 + (e >> 1)];
        x[kc][h][e] = fmaf(st.alpha, x[kc][h][e], (e & 1) ? bf_hi(u) : bf_lo(u));
        ss += x[kc][h][e] * x[kc][h][e];
      }
  ss = wave_sum(ss);
  const float r = 1.f / sqrtf(ss / (float)st.k_real + st.norm_eps);
#pragma unroll
  for (int kc = 0; kc < KL; kc++) {
    u32x4 o16;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] = (x[kc][h][e] * r) * (st.w_offset + g[kc][h][e]);
      o16[h * 2] = pack2(o[0], o[1]);
      o16[h * 2 + 1] = pack2(o[2], o[3]);
      if (c.vid == 0 && st.out2) stc_16B((u32x4 *)st.out2 + (kc * 64 + lane) * 2 + h, __builtin_bit_cast(u32x4, o));
    }
    ((u32x4 *)xs)[kc * 64 + lane] = o16;
    if (c.vid == 0) stc_16B((u32x4 *)st.norm_out + kc * 64 + lane, o16);
  }
}

// Single-token linear: out[n] = bf16(sum_k W[n,k] * x[k] (+ res[n])), optionally with the RMSNorm of x
// fused in front and with the SwiGLU epilogue fused behind.  The weight matrix is streamed from HBM
// exactly once with 128-bit loads, one 1 KB row segment per wavefront instruction; x lives in LDS as
// packed bf16 and the products run on v_dot2_f32_bf16 with fp32 accumulation.
//
// Wavefront roles: wavefront 0 is the control wavefront -- it polls the grid barrier, then loads, normalises and
// publishes x, and only then joins the streaming -- while wavefronts 1..3 stream weight rows from the start.  A
// wavefront's vector loads return in order, so a wavefront that has weight loads in flight cannot observe the
// barrier before they land; keeping the poll on a wavefront without weight loads lets the weight prefetch and the
// barrier overlap.
// KL = K/512 row segments per lane.  Every worker keeps U outputs' rows in flight in registers; the first U are
// requested BEFORE the previous stage is known to be complete (weights do not depend on it), so the HBM pipe stays
// busy across the grid barrier, and a slot is refilled from the workgroup's ticket counter as soon as it is consumed.
// Reference tasks: linear_kernel_ck (tasks/mi300/linear_ck_mi300.cuh:289-619), gang_linear_silu_kernel
// (tasks/mi300/gang_linear_mi300.cuh:359-576).
template <int KL, int R, bool SILU, bool W0OK, bool FX>
__device__ __forceinline__ void stage_linear_m1_t(CStage &st, Ctx &c, char *smem) {
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int K8 = KL * 64;
  constexpr int NROW = SILU ? 2 : 1;  // weight rows per output ([gate ; up] pair)
  constexpr int U = R / NROW;         // outputs in flight per worker wavefront
  uint32_t *xs = (uint32_t *)smem;
  const bool ctrl = wave == 0;
  const int n_out = SILU ? st.n / 2 : st.n;
  // The workgroup owns a contiguous range of outputs; its three worker wavefronts draw them one at a time from an LDS
  // ticket counter, so all three stream until the range is exhausted however the CU's memory pipeline favours them.
  const int oq = n_out / c.G, orem = n_out - oq * c.G;
  const int o_begin = c.vid * oq + min(c.vid, orem), o_end = o_begin + oq + (c.vid < orem ? 1 : 0);
  int *ticket = c.sh_ticket + (c.seq & 1);
  const int half = st.silu_half;
  auto take = [&]() -> int {  // next output index of this workgroup, or -1
    int t = 0;
    if (lane == 0) t = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    t = __builtin_amdgcn_readfirstlane(t) + o_begin;
    return t < o_end ? t : -1;
  };
  auto load_unit = [&](int o, u32x4 (&b)[NROW][KL]) {
    int vr = o;
    if (SILU) {
      const int g = o / half;
      vr = g * 2 * half + (o - g * half);
    }
#pragma unroll
    for (int h = 0; h < NROW; h++) {
      const u32x4 *p = weight_row(st.w, vr + h * half, K8) + lane;
#pragma unroll
      for (int kc = 0; kc < KL; kc++) b[h][kc] = ldg_stream(p + kc * 64);
    }
  };
  u32x4 buf[U][NROW][KL];
  int uo[U];
  // LDS side of the prefetch: NL further outputs per worker wavefront whose rows are parked in the LDS window above
  // MK_MOE_OFFSET while the barrier is awaited (the registers alone hold about 3.5 us of streaming, the barrier and the
  // staging of the input row take longer).  They are reduced from LDS right after the barrier.
  constexpr int NLFIT = 32 / (KL * NROW);  // rows of KL KB that fit a wavefront's 32 KB share of the window
  constexpr int NL = NLFIT < MK_TUNE_NL ? NLFIT : MK_TUNE_NL;
  u32x4 *lrows = (u32x4 *)(smem + MK_MOE_OFFSET) + (size_t)(wave > 0 ? wave - 1 : 0) * (NL > 0 ? NL : 1) * NROW * K8;
  int lo_[NL > 0 ? NL : 1];
  if (!ctrl) {
    // weights do not depend on the previous stage: the first outputs' rows are requested before its barrier completes
    if (NL > 0) {
      // A rolling window of U outputs: output i goes to register slot i % U; from the U-th on, the slot's previous
      // output has landed by then and is parked in LDS first.  The first NL outputs end up parked, the last U stay in the
      // register slots, and never more than U outputs per wavefront are in flight -- a load the control wavefront issues
      // (the barrier poll, then the input row) queues behind whatever the CU has in flight, so it must not be the whole
      // prefetch.  Every load is unconditional (an exhausted ticket re-reads a valid row), so the waits count exactly.
#pragma unroll
      for (int i = 0; i < NL + U; i++) {
        const int sl = i % U;
        if (i >= U) {
#pragma unroll
          for (int h = 0; h < NROW; h++)
#pragma unroll
            for (int kc = 0; kc < KL; kc++) lrows[(((i - U) * NROW + h) * KL + kc) * 64 + lane] = buf[sl][h][kc];
          lo_[i - U] = uo[sl];
        }
        uo[sl] = take();
        load_unit(uo[sl] >= 0 ? uo[sl] : min(o_begin, n_out - 1), buf[sl]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < U; j++) {
        uo[j] = take();
        if (uo[j] >= 0) load_unit(uo[j], buf[j]);
      }
    }
#if MK_HAVE_MIX
  } else if (FX && (st.flags & MK_F_PRENORM)) {
    if constexpr (FX && KL <= 8) mx_x_m1_prenorm_wave<KL>(st, c, xs, lane);
#endif
  } else if (FX && (st.flags & MK_F_ADDNORM)) {
    if constexpr (FX && KL <= 8) stage_x_m1_addnorm_wave<KL>(st, c, xs, lane);  // (longer rows take the generic form)
  } else {
    u32x4 nwv[KL];
    if (st.flags & MK_F_NORM) {
#pragma unroll
      for (int kc = 0; kc < KL; kc++) nwv[kc] = ((const u32x4 *)st.norm_w)[kc * 64 + lane];
    }
    if (c.pending && tid == 0) barrier_poll(c);
    stage_x_m1_wave<KL>(st, c, xs, lane, nwv);
  }
  __syncthreads();
  barrier_done(c);
  // Outputs are collected in LDS and written out together once every worker is done: one write-through request per
  // 128-byte line instead of one 2-byte write per output.
  uint16_t *so = (uint16_t *)(smem + MK_OUT_OFFSET);
  // Rows of 8 KB and more: wavefront 0 alone writes the outputs out, so that the arrival needs no workgroup barrier and
  // the other wavefronts go straight on to the next stage's prefetch (barrier_arrive).  With shorter rows (stages of a
  // few microseconds) the earlier prefetch gains less than it costs wavefront 0's arrival and next poll, which then
  // queue behind it.
  // (only in the kernel instantiation for single-token graphs: W0OK)
  constexpr bool W0 = W0OK && KL >= MK_TUNE_W0_KL;
  auto flush = [&]() {
    if (W0 && tid == 0) c.sh_ticket[(c.seq + 1) & 1] = 0;  // the next stage's work counter (idle since the previous stage)
    __syncthreads();
    uint16_t *dst = (uint16_t *)st.out + o_begin;
    if (W0) {
      if (wave == 0) {
        for (int i = lane; i < o_end - o_begin; i += 64) stc_u16(dst + i, so[i]);
      }
    } else {
      for (int i = tid; i < o_end - o_begin; i += MK_THREADS) stc_u16(dst + i, so[i]);
    }
    c.wrote_through = true;
    c.arrive_w0 = W0;
  };
  if (ctrl) {  // the control wavefront has done its part: it now streams rows like the others
#pragma unroll
    for (int j = 0; j < U; j++) {
      uo[j] = take();
      if (uo[j] >= 0) load_unit(uo[j], buf[j]);
    }
  }
  const bool has_res = st.flags & MK_F_RES;
  const uint16_t *res = (const uint16_t *)st.res;
  float ures[U];
#pragma unroll
  for (int j = 0; j < U; j++) ures[j] = (has_res && uo[j] >= 0) ? bf2f(ldc_u16(res + uo[j])) : 0.f;
  // (the residual values of the parked outputs too: requested together here, not one round trip per parked output)
  float lres[NL > 0 ? NL : 1];
#pragma unroll
  for (int i = 0; i < (NL > 0 ? NL : 1); i++) lres[i] = (NL > 0 && has_res && !ctrl && lo_[i] >= 0) ? bf2f(ldc_u16(res + lo_[i])) : 0.f;
  const u32x4 *xs4 = (const u32x4 *)xs;
  u32x4 xr[KL <= 8 ? KL : 1];
  if (KL <= 8) {
#pragma unroll
    for (int kc = 0; kc < (KL <= 8 ? KL : 1); kc++) xr[kc] = xs4[kc * 64 + lane];
  }
  if (NL > 0 && !ctrl) {  // the parked rows first: no memory traffic, the register slots keep landing meanwhile
#pragma unroll
    for (int i = 0; i < NL; i++) {
      if (lo_[i] >= 0) {
        float a[NROW];
#pragma unroll
        for (int h = 0; h < NROW; h++) {
          a[h] = 0.f;
#pragma unroll
          for (int kc = 0; kc < KL; kc++) a[h] = dot8(lrows[((i * NROW + h) * KL + kc) * 64 + lane], KL <= 8 ? xr[KL <= 8 ? kc : 0] : xs4[kc * 64 + lane], a[h]);
        }
#pragma unroll
        for (int h = 0; h < NROW; h++) a[h] = wave_sum(a[h]);
        const float v = SILU ? linear_glu(st, a[0], a[NROW - 1]) : linear_act(st, a[0] + lres[i]);
        if (lane == 0) so[lo_[i] - o_begin] = (uint16_t)f2bf(v);
      }
    }
  }
  while (true) {
    bool any = false;
#pragma unroll
    for (int j = 0; j < U; j++) {
      if (uo[j] >= 0) {
        any = true;
        float a[NROW];
#pragma unroll
        for (int h = 0; h < NROW; h++) {
          a[h] = 0.f;
#pragma unroll
          for (int kc = 0; kc < KL; kc++) a[h] = dot8(buf[j][h][kc], KL <= 8 ? xr[KL <= 8 ? kc : 0] : xs4[kc * 64 + lane], a[h]);
        }
        const int o = uo[j];
        const float r = ures[j];
        uo[j] = take();
        if (uo[j] >= 0) {
          load_unit(uo[j], buf[j]);
          if (has_res) ures[j] = bf2f(ldc_u16(res + uo[j]));
        }
#pragma unroll
        for (int h = 0; h < NROW; h++) a[h] = wave_sum(a[h]);
        const float v = SILU ? linear_glu(st, a[0], a[NROW - 1]) : linear_act(st, a[0] + r);
        if (lane == 0) so[o - o_begin] = (uint16_t)f2bf(v);
      }
    }
    if (!any) break;
  }
  flush();
}

// Generic single-token linear for reduction lengths that are not a multiple of 512 or have no tuned
// instantiation: same arithmetic, no cross-barrier prefetch.
template <bool FX>
__device__ __forceinline__ void stage_linear_m1_generic(CStage &st, Ctx &c, char *smem) {
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = st.k, k8 = K / 8;
  uint32_t *xs = (uint32_t *)smem;
  float *red = (float *)(smem + MK_RED_OFFSET);
  barrier_wait(c);
  stage_x_m1<FX>(st, c, xs, red);
  const bool silu = st.flags & MK_F_SILU;
  const int n_out = silu ? st.n / 2 : st.n;
  const int nwaves = c.G * MK_WAVES;
  const int rpw = (n_out + nwaves - 1) / nwaves;
  const int r0 = (c.vid * MK_WAVES + wave) * rpw;
  const int r1 = min(n_out, r0 + rpw);
  const u32x4 *xs4 = (const u32x4 *)xs;
  uint16_t *out = (uint16_t *)st.out;
  const uint16_t *res = (const uint16_t *)st.res;
  for (int r = r0; r < r1; r++) {
    float v;
    if (silu) {
      const int half = st.silu_half;
      const int vr = (r / half) * 2 * half + (r % half);
      const u32x4 *wg = weight_row(st.w, vr, k8);
      const u32x4 *wu = weight_row(st.w, vr + half, k8);
      float ag = 0.f, au = 0.f;
#pragma unroll 4
      for (int kc = lane; kc < k8; kc += 64) {
        const u32x4 x = xs4[kc];
        ag = dot8(ldg_stream(wg + kc), x, ag);
        au = dot8(ldg_stream(wu + kc), x, au);
      }
      v = linear_glu(st, wave_sum(ag), wave_sum(au));
    } else {
      const u32x4 *w0 = weight_row(st.w, r, k8);
      float a0 = 0.f;
#pragma unroll 4
      for (int kc = lane; kc < k8; kc += 64) a0 = dot8(ldg_stream(w0 + kc), xs4[kc], a0);
      v = wave_sum(a0);
      if (st.flags & MK_F_RES) v += bf2f(ldc_u16(res + r));
      v = linear_act(st, v);
    }
    if (lane == 0) out[r] = (uint16_t)f2bf(v);
  }
}

template <bool W0OK, bool FX>
__device__ __forceinline__ void stage_linear_m1(CStage &st, Ctx &c, char *smem) {
  const bool silu = st.flags & MK_F_SILU;
  // the tuned forms collect a workgroup's outputs in the LDS window [MK_OUT_OFFSET, MK_MOE_OFFSET)
  const bool fits = ((silu ? st.n / 2 : st.n) / c.G + 1) * 2 <= MK_MOE_OFFSET - MK_OUT_OFFSET;
#if MK_HAVE_MIX
  if (FX && mx_linear_m1_form(st)) {
    stage_mx_linear_m1(st, c, smem);
    return;
  }
#endif
  if (!fits || (FX && (st.flags & MK_F_ADDNORM) && st.k > 4096)) {
    stage_linear_m1_generic<FX>(st, c, smem);
#if MK_HAVE_MIX
  } else if (FX && (st.flags & MK_F_PRENORM) && !mx_prenorm_by_wave(st)) {
    stage_linear_m1_generic<FX>(st, c, smem);
#endif
  } else if (st.k == 4096) {
    if (silu) stage_linear_m1_t<8, MK_TUNE_R8, true, W0OK, FX>(st, c, smem);
    else stage_linear_m1_t<8, MK_TUNE_R8N, false, W0OK, FX>(st, c, smem);
  } else if (st.k == 12288 && !silu) {
    stage_linear_m1_t<24, MK_TUNE_R24, false, W0OK, FX>(st, c, smem);
  } else if (st.k == 2048) {
    if (silu) stage_linear_m1_t<4, 4, true, W0OK, FX>(st, c, smem);
    else stage_linear_m1_t<4, MK_TUNE_R4, false, W0OK, FX>(st, c, smem);
  } else if (st.k == 1024 && !silu) {
    stage_linear_m1_t<2, 4, false, W0OK, FX>(st, c, smem);
  } else {
    stage_linear_m1_generic<FX>(st, c, smem);
  }
}


// Few-token linear (2..MB tokens): the single-token structure with the token rows in LDS.  Every weight row is still
// read once and dotted against all token rows (v_dot2, fp32); up to 8 tokens this stays under the streaming time, so
// small batches cost little more than one token, where the matrix-core path (16-row tiles, one tile per workgroup
// on the narrow stages) is bound by latency.  A stage that carries MK_F_NORM normalises the rows itself while staging
// them (the standalone NORM stage in front is skipped for these batch sizes).  Outputs are collected in LDS
// [token][output] and written through.
template <int KL, int R, bool SILU, int MB>
__device__ __forceinline__ void stage_linear_small(CStage &st, Ctx &c, int M, char *smem) {
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int K8 = KL * 64;
  constexpr int NROW = SILU ? 2 : 1;
  constexpr int U = R / NROW;
  const bool ctrl = wave == 0;
  const int n_out = SILU ? st.n / 2 : st.n;
  const int oq = n_out / c.G, orem = n_out - oq * c.G;
  const int o_begin = c.vid * oq + min(c.vid, orem), o_end = o_begin + oq + (c.vid < orem ? 1 : 0);
  const int n_loc = o_end - o_begin;
  int *ticket = c.sh_ticket + (c.seq & 1);
  const int half = st.silu_half;
  // Plain rows are drawn and reduced two at a time: a token-row segment read from LDS is used for both weight rows
  // (half the LDS reads per output); a [gate ; up] pair already shares the segment.
  constexpr int Q = SILU ? 1 : 2;  // outputs per ticket
  static_assert(U == 2 * Q, "two groups of rows in flight");
  auto take = [&]() -> int {  // first output of the next group of this workgroup (may lie at or beyond o_end)
    int t = 0;
    if (lane == 0) t = __hip_atomic_fetch_add(ticket, Q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    return __builtin_amdgcn_readfirstlane(t) + o_begin;
  };
  auto load_unit = [&](int o, u32x4 (&b)[NROW][KL]) {
    int vr = o;
    if (SILU) {
      const int g = o / half;
      vr = g * 2 * half + (o - g * half);
    }
#pragma unroll
    for (int h = 0; h < NROW; h++) {
      const u32x4 *p = weight_row(st.w, vr + h * half, K8) + lane;
#pragma unroll
      for (int kc = 0; kc < KL; kc++) b[h][kc] = ldg_stream(p + kc * 64);
    }
  };
  // Every load is unconditional: a group at or beyond the end of the range re-reads the range's last row and its
  // results are dropped.  (A load under a branch would turn every wait for one group into a drain of the other too.)
  // The residual values of a group travel with its rows: lane (q * MB + m) loads the one of output q, token m (stages
  // without a residual read a valid dummy location instead, so that this load is unconditional too).
  const bool has_res = st.flags & MK_F_RES;
  const uint16_t *rbase = has_res ? (const uint16_t *)st.res + (size_t)min(lane & (MB - 1), M - 1) * st.ld_res : (const uint16_t *)st.in;
  auto load_group = [&](int o, u32x4 (&b)[Q][NROW][KL], uint16_t &r) {
#pragma unroll
    for (int q = 0; q < Q; q++) load_unit(max(min(o + q, o_end - 1), 0), b[q]);
    r = ldc_half(rbase + (has_res ? max(min(o + ((lane / MB) & (Q - 1)), o_end - 1), 0) : 0));
  };
  u32x4 bufA[Q][NROW][KL], bufB[Q][NROW][KL];
  uint16_t rA = 0, rB = 0;
  int gA = 0, gB = 0;
  if (!ctrl) {
    gA = take();
    load_group(gA, bufA, rA);
    gB = take();
    load_group(gB, bufB, rB);
  } else {
    if (c.pending && tid == 0) barrier_poll(c);
  }
  __syncthreads();
  barrier_done(c);
  // all four wavefronts stage the token rows (the workers' requests queue behind their weight rows, which were issued
  // long before)
  const uint16_t *x = (const uint16_t *)st.in;
  const int ldx = st.ld_in;
  u32x4 *xs4 = (u32x4 *)(smem + MK_MOE_X_OFFSET);  // [token][K8]
  if (st.flags & MK_F_NORM) {
    // Fused RMSNorm (the standalone NORM stage in front is skipped for these batch sizes): every workgroup normalises
    // all rows itself, a wavefront per row, exactly as the single-token form does; virtual workgroup 0 also stores the
    // normalised rows, which are the norm task's output tensor.
    const u32x4 *nw4 = (const u32x4 *)st.norm_w;
    for (int m = wave; m < M; m += MK_WAVES) {
      const auto xr = dev_rows(x + (size_t)m * ldx);
      u32x4 v[KL];
#pragma unroll
      for (int kc = 0; kc < KL; kc++) v[kc] = ldc_16B(xr, (kc * 64 + lane) * 16);
      float ss = 0.f;
#pragma unroll
      for (int kc = 0; kc < KL; kc++) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint32_t u = v[kc][e];
          ss += bf_lo(u) * bf_lo(u) + bf_hi(u) * bf_hi(u);
        }
      }
      ss = wave_sum(ss);
      const float r = rsqrtf(ss / (float)(KL * 512) + st.eps);
      u32x4 *no = (c.vid == 0) ? (u32x4 *)((uint16_t *)st.norm_out + (size_t)m * st.ld_norm) : nullptr;
#pragma unroll
      for (int kc = 0; kc < KL; kc++) {
        const u32x4 g = nw4[kc * 64 + lane];
        u32x4 y;
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = pack2((bf_lo(v[kc][e]) * r) * bf_lo(g[e]), (bf_hi(v[kc][e]) * r) * bf_hi(g[e]));
        xs4[m * K8 + kc * 64 + lane] = y;
        if (no) stc_16B(no + kc * 64 + lane, y);
      }
    }
  } else {
    constexpr int NCH = MB * KL / MK_WAVES;  // 16-byte segments per lane
    u32x4 xv[NCH];
#pragma unroll
    for (int i = 0; i < NCH; i++) {
      const int ci = (i * MK_WAVES + wave) * 64 + lane, m = ci / K8, o = ci - m * K8;
      if (m < M) xv[i] = ldc_16B(dev_rows(x), m * ldx * 2 + o * 16);
    }
#pragma unroll
    for (int i = 0; i < NCH; i++) {
      const int ci = (i * MK_WAVES + wave) * 64 + lane;
      if (ci / K8 < M) xs4[ci] = xv[i];
    }
  }
  __syncthreads();
  if (ctrl) {
    gA = take();
    load_group(gA, bufA, rA);
    gB = take();
    load_group(gB, bufB, rB);
  }
  uint16_t *so = (uint16_t *)smem;  // [token][output - o_begin]
  auto reduce_group = [&](const u32x4 (&b)[Q][NROW][KL], uint16_t r, int o) {
    const float rf = has_res ? bf2f(r) : 0.f;
    // the LDS addresses of the token rows are rebuilt from the lane index in every call: hoisted out of the loop they
    // would be long-lived registers that get spilled, and a spill reload in this loop is a vector-memory wait
    int lo = lane;
    asm volatile("" : "+v"(lo));
    float a[Q][NROW][MB];
    // the segments of token m + 1 are read from LDS while token m is reduced (rows beyond M re-read row M - 1)
    u32x4 xk[2][KL];
#pragma unroll
    for (int kc = 0; kc < KL; kc++) xk[0][kc] = xs4[kc * 64 + lo];
#pragma unroll
    for (int m = 0; m < MB; m++) {
#pragma unroll
      for (int q = 0; q < Q; q++)
#pragma unroll
        for (int h = 0; h < NROW; h++) a[q][h][m] = 0.f;
      if (m + 1 < MB) {
        const int mn = min(m + 1, M - 1);
#pragma unroll
        for (int kc = 0; kc < KL; kc++) xk[(m + 1) & 1][kc] = xs4[mn * K8 + kc * 64 + lo];
      }
      __builtin_amdgcn_sched_barrier(0);
      if (m < M) {
#pragma unroll
        for (int kc = 0; kc < KL; kc++) {
#pragma unroll
          for (int q = 0; q < Q; q++)
#pragma unroll
            for (int h = 0; h < NROW; h++) a[q][h][m] = dot8(b[q][h][kc], xk[m & 1][kc], a[q][h][m]);
        }
      }
    }
    // all Q * NROW * MB sums are reduced together; lane q * MB + m (plain) / h * MB + m ([gate ; up]) gets the total
    constexpr int NV = Q * NROW * MB;
    float vv[NV];
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
      for (int h = 0; h < NROW; h++)
#pragma unroll
        for (int m = 0; m < MB; m++) vv[(q * NROW + h) * MB + m] = a[q][h][m];
    const float tot = transpose_sum<NV>(vv, lane);
    const int m = lane & (MB - 1), q = SILU ? 0 : lane / MB;
    float v;
    if (SILU) v = linear_glu(st, tot, dpp_f32<0x100 + MB>(tot));  // row_shl:MB: the up sum sits MB lanes above the gate sum
    else v = linear_act(st, tot + rf);
    if (lane < Q * MB && m < M && o + q < o_end) so[m * n_loc + (o + q - o_begin)] = (uint16_t)f2bf(v);
  };
  // two groups in flight: while one is reduced the other one's rows are landing; tickets only grow, so the first
  // group found beyond the range ends the loop
  while (gA < o_end) {
    reduce_group(bufA, rA, gA);
    gA = take();
    load_group(gA, bufA, rA);
    if (gB >= o_end) break;
    reduce_group(bufB, rB, gB);
    gB = take();
    load_group(gB, bufB, rB);
  }
  __syncthreads();
  uint16_t *dst = (uint16_t *)st.out + o_begin;
  for (int i = tid; i < M * n_loc; i += MK_THREADS) {
    const int m = i / n_loc, r = i - m * n_loc;
    stc_u16(dst + (size_t)m * st.ld_out + r, so[i]);
  }
  c.wrote_through = true;
}

// Whether the few-token form can run this stage: reduction length with a tuned instantiation, token rows within the
// LDS window above MK_MOE_X_OFFSET, collected outputs within the window below MK_MOE_OFFSET.
#ifndef MK_TUNE_SMALL_MAX
#define MK_TUNE_SMALL_MAX 2
#endif
__device__ __forceinline__ bool linear_small_ok(CStage &st, const Ctx &c, int M) {
  if (M > MK_TUNE_SMALL_MAX || (st.k != 4096 && st.k != 2048) || (st.flags & (MK_F_ADDNORM | MK_F_PRENORM))) return false;
  const int n_out = (st.flags & MK_F_SILU) ? st.n / 2 : st.n;
  return (size_t)M * st.k * 2 <= (size_t)(MK_LDS_BYTES - MK_MOE_X_OFFSET) && (size_t)M * (n_out / c.G + 1) * 2 <= (size_t)MK_MOE_OFFSET;
}

template <int MB>
__device__ __forceinline__ void stage_linear_small_dispatch(CStage &st, Ctx &c, int M, char *smem) {
  const bool silu = st.flags & MK_F_SILU;
  if (st.k == 4096) {
    if (silu) stage_linear_small<8, 4, true, MB>(st, c, M, smem);
    else stage_linear_small<8, 4, false, MB>(st, c, M, smem);
  } else {
    if (silu) stage_linear_small<4, 4, true, MB>(st, c, M, smem);
    else stage_linear_small<4, 4, false, MB>(st, c, M, smem);
  }
}

// Matrix-core linear for several tokens.  A workgroup owns a range of 16-row weight tiles and one K slice (S slices
// per range when a stage has too few tiles to fill the machine, S = 1 otherwise).  The range is worked off in sweeps:
// every wavefront holds TW tiles of the sweep over the whole slice, and all four share the token rows of the slice,
// which one pass stages per 64-wide step in LDS (double-buffered, in matrix-core operand order, so the reads are linear
// in the lane index).  Token-row traffic per weight byte is M / (64 TW); weight steps sit NB deep in registers.
//
// Every load is unconditional and the step loop has a fixed trip structure (slices are multiples of NB steps; slots
// past the range re-read its last tile): a load under a branch makes the compiler's wait counts drain everything
// younger, which costs the whole prefetch depth.  Loads return in issue order, so token rows are prefetched exactly as
// deep as the weights.
//
// With S > 1 the partial tiles go through a write-through buffer; the last workgroup of a group to arrive sums them in
// slice order (deterministic), applies SwiGLU / residual and stores bf16.  SwiGLU stages number their weight tiles
// gate, up, gate, up ... so that a pair always sits in one wavefront.
// Reference tasks: linear / linear_with_residual / splitk_linear (tasks/mi300/linear_ck_mi300.cuh), silu_mul_linear.
#ifndef MK_TUNE_SPLITK_MAXS
#define MK_TUNE_SPLITK_MAXS 8
#endif
#ifndef MK_TUNE_TPU
#define MK_TUNE_TPU 4  // tiles per workgroup a split stage aims for
#endif
#ifndef MK_TUNE_NB1
#define MK_TUNE_NB1 8
#endif
#ifndef MK_TUNE_NB2
#define MK_TUNE_NB2 4
#endif
#ifndef MK_TUNE_NB4
#define MK_TUNE_NB4 2
#endif
#ifndef MK_TUNE_TILES_MIN_TPW
#define MK_TUNE_TILES_MIN_TPW 16
#endif
#define MK_TILES_NB 4  // a K slice is a multiple of 64 * 2 * MK_TILES_NB (the deepest instantiation's ring)

struct TilePlan {
  int S;       // K slices per tile range (0: this form cannot run the stage)
  int groups;  // tile ranges
  int wt;      // weight tiles of the stage
};
__device__ __forceinline__ TilePlan linear_tiles_plan(CStage &st, const Ctx &c) {
  TilePlan p;
  const bool silu = st.flags & MK_F_SILU;
  const int n_out = silu ? st.n / 2 : st.n;
  const int unit = silu ? 2 : 1;                      // ranges are made of whole gate/up pairs
  p.wt = ((n_out + 15) / 16) * unit;
  p.S = 0;
  p.groups = 0;
  if (st.k % (64 * 2 * MK_TILES_NB) != 0) return p;
  const int tpw = (p.wt + c.G - 1) / c.G;            // tiles per workgroup without a K split
  int S = 1;
  while (S < MK_TUNE_SPLITK_MAXS && tpw * S < MK_TUNE_TPU && 2 * S <= c.G && st.k % (S * 2 * 64 * 2 * MK_TILES_NB) == 0) S *= 2;
  const int gs = c.G / S;                             // ranges the grid can hold: S adjacent workgroups each
  int tpu = (p.wt + gs - 1) / gs;                     // tiles per range
  tpu = (tpu + unit - 1) / unit * unit;
  if (S > 1 && tpu > 16) return p;                    // a split range is a single sweep
  if (S == 1 && tpw < MK_TUNE_TILES_MIN_TPW) return p;  // a few tiles per workgroup without a K split: the form that splits K inside the workgroup
  p.groups = (p.wt + tpu - 1) / tpu;
  p.S = S;
  return p;
}

template <int MT>
__device__ __forceinline__ void stage_linear_mfma_tiles(CStage &st, Ctx &c, const MkRuntime &rt, int M, const TilePlan plan, char *smem) {
  barrier_wait(c);
  c.wrote_through = true;  // partial tiles and outputs are all written through: no L2 write-back at this stage's arrival
  MK_MARK(c, 0);
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const bool silu = st.flags & MK_F_SILU;
  const int K = st.k, k8 = K / 8;
  const int n_out = silu ? st.n / 2 : st.n;
  const int half = st.silu_half;
  const int S = plan.S, unit = silu ? 2 : 1;
  const int g = c.vid / S, sl = c.vid - g * S;
  if (g >= plan.groups) return;  // workgroups beyond the last range have nothing to do in this stage
  // balanced ranges of whole units
  const int nun = plan.wt / unit;
  const int tb = (int)(((long long)g * nun) / plan.groups) * unit, te = (int)(((long long)(g + 1) * nun) / plan.groups) * unit;
  const int kslice = K / S, kbeg = sl * kslice, nsteps = kslice >> 6;
  const uint16_t *x = (st.flags & MK_F_NORM) ? (const uint16_t *)st.norm_out : (const uint16_t *)st.in;
  const int ldx = (st.flags & MK_F_NORM) ? st.ld_norm : st.ld_in;
  u32x4 *xl = (u32x4 *)smem;  // two buffers of [MT][2][64] 16-byte operands
  int *sflag = (int *)(smem + 2 * MT * 2048);
  // token rows: wavefront w stages token tile w, every lane the same 32 contiguous bytes it would feed the matrix core
  // with, stored at its own lane slot of the operand block (consecutive 16-byte slots: no bank conflicts either way)
  const auto xrows = dev_rows(x);
  const int xsrc = (min(min(wave, MT - 1) * 16 + lr, M - 1) * ldx + kbeg + lg * 16) * 2;  // bytes
  const int xdst = min(wave, MT - 1) * 128 + lane;
  // first weight row of weight tile ti for this lane
  auto tile_row = [&](int ti) -> const uint16_t * {
    int o, vr;
    if (silu) {
      o = min((ti >> 1) * 16 + lr, n_out - 1);
      const int gi = o / half;
      vr = gi * 2 * half + (o - gi * half) + ((ti & 1) ? half : 0);
    } else {
      o = min(ti * 16 + lr, n_out - 1);
      vr = o;
    }
    return (const uint16_t *)weight_row(st.w, vr, k8) + kbeg + lg * 16;
  };
  u32x4 *part = (u32x4 *)rt.splitk_part;

  auto sweep = [&](int t0, auto twc) {
    constexpr int TW = decltype(twc)::value;
    constexpr int NB = TW == 1 ? MK_TUNE_NB1 : (TW == 2 ? MK_TUNE_NB2 : MK_TUNE_NB4);
    const int tw0 = t0 + wave * TW;           // this wavefront's first tile
    const bool has_tile = tw0 < te;           // wavefronts without one only stage token rows and keep the barriers
    const uint16_t *wrow[TW];
#pragma unroll
    for (int t = 0; t < TW; t++) wrow[t] = tile_row(min(tw0 + t, te - 1));
    bf16x8 a[NB][TW][2];
    u32x4 xq[NB][2];
    auto w_load = [&](int step, bf16x8 (&aa)[TW][2]) {
#pragma unroll
      for (int t = 0; t < TW; t++) {
        aa[t][0] = __builtin_nontemporal_load((const bf16x8 *)(wrow[t] + (step << 6)));
        aa[t][1] = __builtin_nontemporal_load((const bf16x8 *)(wrow[t] + (step << 6) + 8));
      }
    };
    auto x_load = [&](int step, u32x4 (&q)[2]) {
      q[0] = ldc_16B(xrows, xsrc + (step << 7));
      q[1] = ldc_16B(xrows, xsrc + (step << 7) + 16);
    };
    auto x_store = [&](int buf, const u32x4 (&q)[2]) {
      if (wave < MT) {
        xl[buf * MT * 128 + xdst] = q[0];
        xl[buf * MT * 128 + xdst + 64] = q[1];
      }
    };
    f32x4 acc[TW][MT];
#pragma unroll
    for (int t = 0; t < TW; t++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) acc[t][mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // Copies of the step loop for wavefronts with / without tiles and with / without a token tile to stage: a branch
    // around loads inside one copy would spoil its wait counts.  All copies execute the same barriers.
    auto pipeline = [&](auto htc, auto xlc) {
      constexpr bool HT = decltype(htc)::value;
      constexpr bool XL = decltype(xlc)::value;  // this wavefront stages a token tile (wavefront index < MT)
      __syncthreads();  // the previous sweep has finished with the LDS buffers
#pragma unroll
      for (int j = 0; j < NB; j++) {
        if (HT) w_load(j, a[j]);
        if (XL) x_load(j, xq[j]);
      }
      if (XL) x_store(0, xq[0]);
      __syncthreads();
      auto block = [&](int s0, auto refill) {
        constexpr bool REFILL = decltype(refill)::value;
#pragma unroll
        for (int j = 0; j < NB; j++) {
          const int step = s0 + j;
          if (XL && (REFILL || j + 1 < NB)) x_store((step + 1) & 1, xq[(j + 1) % NB]);  // that buffer was last read before the previous barrier
          if (HT) {
            const u32x4 *xb = xl + (step & 1) * MT * 128;
            u32x4 b[2][MT];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
              for (int mt = 0; mt < MT; mt++) b[h][mt] = xb[(mt * 2 + h) * 64 + lane];
            __builtin_amdgcn_sched_barrier(0);  // all operand reads in flight before the first matrix instruction waits
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
              for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int t = 0; t < TW; t++)
                  acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j][t][h], __builtin_bit_cast(bf16x8, b[h][mt]), acc[t][mt], 0, 0, 0);
          }
          if (REFILL) {
            if (HT) w_load(step + NB, a[j]);
            if (XL) x_load(step + NB, xq[j]);
          }
          __syncthreads();
        }
      };
      int s0 = 0;
      for (; s0 + NB < nsteps; s0 += NB) block(s0, std::true_type{});
      block(s0, std::false_type{});
    };
    const bool stages_x = wave < MT;
    if (MT == MK_WAVES || stages_x) {
      if (has_tile) pipeline(std::true_type{}, std::true_type{});
      else pipeline(std::false_type{}, std::true_type{});
    } else {
      if (has_tile) pipeline(std::true_type{}, std::false_type{});
      else pipeline(std::false_type{}, std::false_type{});
    }

    MK_MARK(c, 1);
    // ---- combine the S slices (a split range is a single sweep, so slots are indexed by wavefront and tile only)
    if (S > 1) {
      if (has_tile) {
#pragma unroll
        for (int t = 0; t < TW; t++)
#pragma unroll
          for (int mt = 0; mt < MT; mt++)
            stc_16B(part + ((((size_t)c.vid * 4 + wave) * 4 + t) * 4 + mt) * 64 + lane, __builtin_bit_cast(u32x4, acc[t][mt]));
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) {
        unsigned *cnt = rt.splitk_cnt + (size_t)g * 32;
        const int last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(S - 1);
        if (last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *sflag = last;
      }
      __syncthreads();
      MK_MARK(c, 2);
      if (!*sflag || !has_tile) return;
#pragma unroll
      for (int t = 0; t < TW; t++) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[t][mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
        for (int q0 = 0; q0 < S; q0 += 4) {  // four slices requested at once; summed in slice order
          u32x4 pv[4][MT];
#pragma unroll
          for (int q = 0; q < 4; q++)
            if (q0 + q < S) {
#pragma unroll
              for (int mt = 0; mt < MT; mt++) pv[q][mt] = ldc_16B(part + ((((size_t)(g * S + q0 + q) * 4 + wave) * 4 + t) * 4 + mt) * 64 + lane);
            }
#pragma unroll
          for (int q = 0; q < 4; q++)
            if (q0 + q < S) {
#pragma unroll
              for (int mt = 0; mt < MT; mt++) acc[t][mt] += __builtin_bit_cast(f32x4, pv[q][mt]);
            }
        }
      }
    }
    MK_MARK(c, 3);
    if (!has_tile) return;
    // ---- epilogue: lane l holds token m = mt * 16 + (l & 15), output columns tile * 16 + (l >> 4) * 4 .. + 3
    constexpr int OT = TW >= 2 ? TW / 2 : 1;
#pragma unroll
    for (int u = 0; u < (TW >= 2 ? TW : 1); u++) {
      if (silu && u >= OT) break;
      const int ti = silu ? tw0 + 2 * u : tw0 + u;
      if (ti >= te) break;
      const int otile = silu ? (ti >> 1) : ti;
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        const int m = mt * 16 + lr;
        if (m < M) {
          uint16_t *orow = (uint16_t *)st.out + (size_t)m * st.ld_out;
          const uint16_t *rrow = (const uint16_t *)st.res + (size_t)m * st.ld_res;
          float rr[4], res[4];
          if (st.flags & MK_F_RES) ldc_bf16x4(rrow, otile * 16 + lg * 4, n_out, res);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            float r;
            if (silu) r = TW >= 2 ? linear_glu(st, acc[(2 * u) % TW][mt][i], acc[(2 * u + 1) % TW][mt][i]) : 0.f;
            else r = acc[u][mt][i];
            if (st.flags & MK_F_RES) r += res[i];
            rr[i] = linear_act(st, r);
          }
          stc_bf16x4(orow, otile * 16 + lg * 4, n_out, rr);
        }
      }
    }
  };

  for (int t0 = tb; t0 < te;) {
    const int r = te - t0;
    if (r > 8) {
      sweep(t0, std::integral_constant<int, 4>{});
      t0 += 16;
    } else if (r > 4 || silu) {
      sweep(t0, std::integral_constant<int, 2>{});
      t0 += 8;
    } else {
      sweep(t0, std::integral_constant<int, 1>{});
      t0 += 4;
    }
  }
}

// Matrix-core linear with the token rows staged through LDS by wavefronts of their own.  A workgroup owns a range of 4..6
// weight tiles and one K slice, which it works off in passes of 8 steps (512 k).  Wavefronts 0 and 1 hold two or three
// tiles each and do nothing but stream weights (a ring of NB = 8 steps, 32 or 48 KB per wavefront, which runs on across
// the passes without ever draining) and feed the matrix cores from LDS; wavefronts 2 and 3 stage the token rows of the
// NEXT pass -- all rows, 64 KB for 64 tokens, in matrix-core operand order, with loads that write LDS directly (no
// registers) -- into the other half of a double buffer.  Loads return in issue order per wavefront, and a token-row
// load queues behind the weight stream in the memory system like any other request, so in a wavefront that also
// streams weights every batch of row loads stalls the weight ring for a full memory latency; on wavefronts of their
// own they cost the streaming wavefronts nothing.  (One staging wavefront is not enough: with at most 63 requests
// outstanding it needs two memory latencies for the 128 requests of a pass, and the pass cannot be shorter than that.)
// One workgroup barrier per pass hands a buffer over.  The first NB weight steps are requested before the previous
// stage's barrier is awaited; the rows of the first pass are staged by all four wavefronts.  The S workgroups that
// share a tile range exchange their partial tiles as the streaming form does (write-through buffer, last arriver sums
// in slice order), or leave the sum to a norm stage that follows.  Used for the QKV, o, gate/up and down projections at
// 9..64 tokens.  SwiGLU stages number their weight tiles gate, up, gate, up ...; with three tiles per wavefront the
// middle pair straddles the two streaming wavefronts and is joined through LDS in the epilogue.
#ifndef MK_TUNE_XRES_PRE
#define MK_TUNE_XRES_PRE 6  // ring steps requested before the previous stage's barrier is awaited
#endif
__device__ __forceinline__ XresPlan linear_xres_plan(CStage &st, const Ctx &c) { return mk_xres_plan(st, c.G); }

// MT token tiles.
template <int MT, int TW>
__device__ __forceinline__ void stage_linear_mfma_xres(CStage &st, Ctx &c, const MkRuntime &rt, int M, const XresPlan plan, char *smem) {
  c.wrote_through = true;  // partial tiles and outputs are all written through: no L2 write-back at this stage's arrival
  constexpr int NSP = MK_XRES_STEPS;
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const bool silu = st.flags & MK_F_SILU;
  const int K = st.k, k8 = K / 8;
  const int n_out = silu ? st.n / 2 : st.n, unit = silu ? 2 : 1;
  const int half = st.silu_half;
  const int S = plan.S;
  const int g = c.vid / S, sl = c.vid - g * S;
  // ranges [q0, q0 + nr) of this workgroup; workgroups beyond the last range only keep the barriers
  const int q0 = plan.R > 1 ? (int)(((long long)c.vid * plan.groups) / c.G) : g, nr = plan.R > 1 ? (int)(((long long)(c.vid + 1) * plan.groups) / c.G) - q0 : (g < plan.groups ? 1 : 0);
  const bool active = nr > 0;
  const int nun = plan.wt / unit;  // balanced ranges of whole units
  auto range_at = [&](int q) { return (int)(((long long)q * nun) / plan.groups) * unit; };
  int tb = active ? range_at(q0) : 0, te = active ? range_at(q0 + 1) : 0;
  const int kslice = K / S, kbeg = sl * kslice, nsteps = kslice >> 6, npass = nsteps / NSP;
  const uint16_t *x = (st.flags & MK_F_NORM) ? (const uint16_t *)st.norm_out : (const uint16_t *)st.in;
  const int ldx = (st.flags & MK_F_NORM) ? st.ld_norm : st.ld_in;
  u32x4 *xl = (u32x4 *)smem;  // two buffers of [step of the pass][token tile][16 rows][8] 16-byte words
  constexpr int XBUF = NSP * MT * 128;  // 16-byte operands per buffer
  int *sflag = (int *)(smem + 2 * XBUF * 16);
  u32x4 *xpair = xl + 2 * XBUF + 16;  // a gate/up pair that two wavefronts hold
  u32x4 *part = (u32x4 *)rt.splitk_part;
  // hand the K-slice sum to the norm stage that follows, if there is one and the rows fit the partial buffer
  bool defer = (st.flags & MK_F_DEFER_SUM) && S > 1 && (size_t)S * (MT * 16) * st.n * 4 <= (size_t)c.G * 65536;
#if MK_PAIR
  defer = defer && !c.keeps_sum;
#endif
  if (defer) {
    c.defer_S = S;
    c.defer_rows = MT * 16;
    c.defer_n = st.n;
    c.defer_part = (const float *)rt.splitk_part;
    c.defer_res = (st.flags & MK_F_RES) ? st.res : nullptr;
    c.defer_ld_res = st.ld_res;
  }
  // this lane's first operand of weight tile ti, and the distance (in 16-byte operands) between steps and between the two
  // halves of a step: the re-laid copy streams contiguously, the row-major original reads 64 bytes of each of 16 rows
  const bool packed = st.wpack != nullptr;
  const int step_stride = packed ? 128 : 8, half_stride = packed ? 64 : 4;
  auto tile_base = [&](int ti) -> const u32x4 * {
    if (packed) return (const u32x4 *)st.wpack + ((size_t)ti * (K >> 6) + (kbeg >> 6)) * 128 + lane;
    int o, vr;
    if (silu) {
      o = min((ti >> 1) * 16 + lr, n_out - 1);
      const int gi = o / half;
      vr = gi * 2 * half + (o - gi * half) + ((ti & 1) ? half : 0);
    } else {
      o = min(ti * 16 + lr, n_out - 1);
      vr = o;
    }
    return weight_row(st.w, vr, k8) + (kbeg >> 3) + lg;
  };
  // stage the token rows of one pass: item i = (step, token tile), two 1 KB requests each, straight into LDS (lane l's 16
  // bytes land at l * 16 behind the request's LDS base).  A request reads whole 128-byte lines of eight rows: in operand order,
  // neighbouring lanes in different rows, a CU takes in 16 bytes a clock, a quarter of what it can.  Word c of row r lies at
  // 8 r + (c ^ (r & 7)), so that the operand reads meet no bank twice.  `nw` wavefronts share the items: wavefront `w` of them takes
  // items w, w + nw, ...
  // (64 tokens, operand order -> lines, us: 24576 x 4096 41.9 -> 39.6, 4096 x 12288 28.9 -> 27.0, 6144 x 4096 17.3 -> 16.7.)
  auto stage_pass = [&](int pass, int par, int w, int nw) {
    const uint16_t *base = x + kbeg + pass * (NSP * 64) + ((lane & 7) ^ (lane >> 3)) * 8;
    u32x4 *buf = xl + (par & 1) * XBUF;
    for (int i = w; i < MT * NSP; i += nw) {
      const int step = i / MT, mt = i - step * MT, r0 = mt * 16 + (lane >> 3);
      __attribute__((address_space(3))) char *dst = (__attribute__((address_space(3))) char *)(buf + (size_t)i * 128);
      __builtin_amdgcn_global_load_lds((const MK_GLOBAL void *)(unsigned long long)(base + (size_t)min(r0, M - 1) * ldx + (step << 6)), (__attribute__((address_space(3))) void *)dst, 16, 0, 16 /* sc1 */);
      __builtin_amdgcn_global_load_lds((const MK_GLOBAL void *)(unsigned long long)(base + (size_t)min(r0 + 8, M - 1) * ldx + (step << 6)), (__attribute__((address_space(3))) void *)(dst + 1024), 16, 0, 16);
    }
  };

  {
    constexpr int NB = NSP, NSW = 2;  // ring depth in steps; streaming wavefronts
    const bool loader = wave >= NSW;  // stages token rows, holds no tiles
    int tw0 = tb + wave * TW;         // a streaming wavefront's first tile
    // (between two ranges of a workgroup the ring stays full, so a wavefront without a tile in one of them reads the last one along)
    const bool streams = active && !loader && (nr > 1 || tw0 < te);
    const u32x4 *wrow[TW];
#pragma unroll
    for (int t = 0; t < TW; t++) wrow[t] = tile_base(max(min(tw0 + t, te - 1), 0));
    bf16x8 a[NB][TW][2];
    auto w_load = [&](const u32x4 *const (&row)[TW], int step, bf16x8 (&aa)[TW][2]) {
#pragma unroll
      for (int t = 0; t < TW; t++) {
        aa[t][0] = __builtin_nontemporal_load((const bf16x8 *)(row[t] + step * step_stride));
        aa[t][1] = __builtin_nontemporal_load((const bf16x8 *)(row[t] + step * step_stride + half_stride));
      }
    };
    // weights do not depend on the previous stage: the first NBP steps are requested before its barrier is awaited, the
    // rest of the ring right after the first pass's token rows (what a CU has in flight sits in front of the barrier
    // poll and of the row requests)
    constexpr int NBP = MK_TUNE_XRES_PRE < NB ? MK_TUNE_XRES_PRE : NB;
    if (streams) {
#pragma unroll
      for (int j = 0; j < NBP; j++) w_load(wrow, j, a[j]);
    }
    // The poll runs on the first row-staging wavefront, which has no weight loads in flight: loads return in order, so
    // on a streaming wavefront the poll's answer would wait behind the NB steps just requested -- two to four
    // microseconds for exactly the workgroups that enter last (those that did the norm stage's rows, or everybody after
    // an attention stage), which are the ones the stage then waits for.
    constexpr int POLL_TID = NSW * 64;
    if (c.pending && tid == POLL_TID) barrier_poll(c);
    __syncthreads();
    barrier_done(c);
    MK_MARK(c, 0);
    f32x4 acc[TW][MT];
    auto compute = [&](const u32x4 *xb, const bf16x8 (&aa)[TW][2]) {
      u32x4 b[2][MT];
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) b[h][mt] = xb[mt * 128 + lr * 8 + ((h * 4 + lg) ^ (lr & 7))];
      __builtin_amdgcn_sched_barrier(0);  // all operand reads in flight before the first matrix instruction waits
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int t = 0; t < TW; t++) acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aa[t][h], __builtin_bit_cast(bf16x8, b[h][mt]), acc[t][mt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    // All passes but the very last one refill the ring as they go, the last of a range with the first steps of the next range.  Every
    // pass starts with a workgroup barrier: its rows have landed (whoever requested them has waited for them) and everybody is done with
    // the other buffer, into which the loader then requests the next pass's rows.
    const u32x4 *wnext[TW];
    int par = 0;  // passes done
    auto do_pass = [&](int pass, auto refill_c) {
      constexpr bool REFILL = decltype(refill_c)::value;
      if (par == 0 && streams && NBP < NB) {
        // the token rows of pass 0 have landed once nothing but the ring steps requested after them is outstanding
        static_assert((NB - NBP) * TW * 2 <= 63, "vmcnt range");
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - NBP) * TW * 2) : "memory");
      } else if (par == 0 || loader) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      lds_barrier();
      if (par == 0) MK_MARK(c, 1);
      const bool in_range = pass + 1 < npass;
      if (loader && active && REFILL) stage_pass(in_range ? pass + 1 : 0, par + 1, wave - NSW, MK_WAVES - NSW);
      __builtin_amdgcn_sched_barrier(0);
      if (streams) {
        const u32x4 *xb = xl + (par & 1) * XBUF;
        static_assert(NB == NSP, "a refill is the same step of the next pass");
        const u32x4 *wr[TW];
#pragma unroll
        for (int t = 0; t < TW; t++) wr[t] = in_range ? wrow[t] : wnext[t];
        const int s0 = in_range ? (pass + 1) * NSP : 0;
#pragma unroll
        for (int j = 0; j < NSP; j++) {
          compute(xb + j * MT * 128, a[j]);
          if (REFILL) w_load(wr, s0 + j, a[j]);
        }
      }
      par++;
    };
    if (active) stage_pass(0, 0, wave, MK_WAVES);
    __builtin_amdgcn_sched_barrier(0);
    if (streams) {
#pragma unroll
      for (int j = NBP; j < NB; j++) w_load(wrow, j, a[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
    auto clear = [&]() {
#pragma unroll
      for (int t = 0; t < TW; t++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[t][mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    };
    // ---- epilogue of a range: lane l holds token m = mt * 16 + (l & 15), output columns tile * 16 + (l >> 4) * 4 .. + 3
    auto finish = [&]() {
      const bool has_tile = active && !loader && tw0 < te;
      if (silu && (TW & 1)) {
        // an odd tile count per wavefront leaves the middle gate/up pair split: wavefront 1 hands its first tile (an up
        // tile) to wavefront 0, which holds the gate tile, through LDS
        if (wave == 1 && has_tile) {
#pragma unroll
          for (int mt = 0; mt < MT; mt++) xpair[mt * 64 + lane] = __builtin_bit_cast(u32x4, acc[0][mt]);
        }
        __syncthreads();
      }
      auto store_tile = [&](int otile, const f32x4 (&v)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
          const int m = mt * 16 + lr;
          if (m < M) {
            uint16_t *orow = (uint16_t *)st.out + (size_t)m * st.ld_out;
            const uint16_t *rrow = (const uint16_t *)st.res + (size_t)m * st.ld_res;
            float rr[4], res[4];
            if (st.flags & MK_F_RES) ldc_bf16x4(rrow, otile * 16 + lg * 4, n_out, res);
#pragma unroll
            for (int i = 0; i < 4; i++) {
              float r = v[mt][i];
              if (st.flags & MK_F_RES) r += res[i];
              rr[i] = linear_act(st, r);
            }
            stc_bf16x4(orow, otile * 16 + lg * 4, n_out, rr);
          }
        }
      };
      if (!has_tile) {
        // (no tile in this range)
      } else if (!silu) {
#pragma unroll
        for (int t = 0; t < TW; t++)
          if (tw0 + t < te) store_tile(tw0 + t, acc[t]);
      } else {
        // tile index relative to the range start is even for gate tiles (ranges hold whole pairs)
#pragma unroll
        for (int t = 0; t < TW; t++) {
          const int ti = tw0 + t;
          if (ti >= te || ((ti - tb) & 1)) continue;  // pairs are stored by the holder of their gate tile
          f32x4 v[MT];
          if (t + 1 < TW) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
              for (int i = 0; i < 4; i++) v[mt][i] = linear_glu(st, acc[t][mt][i], acc[(t + 1) % TW][mt][i]);
          } else {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
              const f32x4 up = __builtin_bit_cast(f32x4, xpair[mt * 64 + lane]);
#pragma unroll
              for (int i = 0; i < 4; i++) v[mt][i] = linear_glu(st, acc[t][mt][i], up[i]);
            }
          }
          store_tile(ti >> 1, v);
        }
      }
    };
    int pass = 0;
    for (int r = 1; r < nr; r++) {  // all ranges but the last
      const int nb_ = range_at(q0 + r), ne_ = range_at(q0 + r + 1);
#pragma unroll
      for (int t = 0; t < TW; t++) wnext[t] = tile_base(min(nb_ + wave * TW + t, ne_ - 1));
      clear();
      for (pass = 0; pass < npass; pass++) do_pass(pass, std::true_type{});
      finish();
      tb = nb_;
      te = ne_;
      tw0 = tb + wave * TW;
#pragma unroll
      for (int t = 0; t < TW; t++) wrow[t] = wnext[t];
    }
#pragma unroll
    for (int t = 0; t < TW; t++) wnext[t] = wrow[t];
    clear();
    for (pass = 0; pass < npass - 1; pass++) do_pass(pass, std::true_type{});
    MK_MARK(c, 2);
    do_pass(pass, std::false_type{});
    MK_MARK(c, 3);
    const bool has_tile = active && !loader && tw0 < te;
    if (defer) {
      // the consumer sums the slices: leave them as [slice][token][n] fp32 rows
      if (has_tile) {
        float *prow = (float *)rt.splitk_part + (size_t)sl * (MT * 16) * st.n;
#pragma unroll
        for (int t = 0; t < TW; t++)
          if (tw0 + t < te) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
              stc_16B((u32x4 *)(prow + (size_t)(mt * 16 + lr) * st.n + (tw0 + t) * 16 + lg * 4), __builtin_bit_cast(u32x4, acc[t][mt]));
          }
      }
      return;
    }
    // ---- combine the S slices: partial tiles through the write-through buffer, summed by the last workgroup to arrive
    if (S > 1) {
      auto part_at = [&](int wg, int ti, int mt) { return ((((size_t)wg * 4 + wave) * 4 + ti) * 4 + mt) * 64 + lane; };
      constexpr int QS = 4;  // slices requested at once
      if (has_tile) {
#pragma unroll
        for (int t = 0; t < TW; t++)
#pragma unroll
          for (int mt = 0; mt < MT; mt++)
            stc_16B(part + part_at(c.vid, t, mt), __builtin_bit_cast(u32x4, acc[t][mt]));
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) {
        int last = 0;
        if (active) {
          unsigned *cnt = rt.splitk_cnt + (size_t)g * 32;
          last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(S - 1);
          if (last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        *sflag = last;
      }
      __syncthreads();
      if (!*sflag) return;  // (the whole workgroup)
#pragma unroll
      for (int t = 0; t < TW; t++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[t][mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
      for (int q0 = 0; has_tile && q0 < S; q0 += QS) {  // summed in slice order
        u32x4 pv[QS][TW][MT];
#pragma unroll
        for (int q = 0; q < QS; q++)
          if (q0 + q < S) {
#pragma unroll
            for (int t = 0; t < TW; t++)
#pragma unroll
              for (int mt = 0; mt < MT; mt++) pv[q][t][mt] = ldc_16B(part + part_at(g * S + q0 + q, t, mt));
          }
#pragma unroll
        for (int q = 0; q < QS; q++)
          if (q0 + q < S) {
#pragma unroll
            for (int t = 0; t < TW; t++)
#pragma unroll
              for (int mt = 0; mt < MT; mt++) acc[t][mt] += __builtin_bit_cast(f32x4, pv[q][t][mt]);
          }
      }
    }
    finish();
  }
}

#ifndef MK_TUNE_NBN
#define MK_TUNE_NBN 4
#endif
// Multi-token linear on the matrix cores, K split inside the workgroup: out[m, n] = bf16(sum_k x[m,k] * W[n,k] (+ res[m,n])) for 2..64 token rows,
// optional SwiGLU epilogue.  A workgroup owns a contiguous range of 16-row weight tiles and ALL token rows, so every
// weight byte is still read from HBM exactly once; its four wavefronts split K and are reduced through LDS.  One
// v_mfma_f32_16x16x32_bf16 consumes a 16(n) x 32(k) weight fragment (one 16-byte load per lane, 64 contiguous bytes per
// weight row) against a 32(k) x 16(m) activation fragment that comes from the L2-resident activation rows.
// Reference tasks: linear_kernel_ck tile tiers (tasks/mi300/linear_ck_mi300.cuh:306-332), gang_linear_kernel
// (tasks/mi300/gang_linear_mi300.cuh:47-108), gang_linear_silu_kernel (:359-576).
// TG = weight tiles per K sweep, NB = 64-wide k steps in flight per wavefront.  Two shapes are instantiated: wide
// stages (several tiles per workgroup) run <6, 2>; narrow ones (one or two weight tiles per workgroup, e.g. N = 4096
// on 256 workgroups) spend the registers on depth instead: <2, MK_TUNE_NBN>.
template <int MT, int TG, int NB>
__device__ __forceinline__ void stage_linear_mfma(CStage &st, Ctx &c, int M, char *smem) {
  barrier_wait(c);
  c.wrote_through = true;  // outputs are written through: no L2 write-back at this stage's arrival
  MK_MARK(c, 0);
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const bool silu = st.flags & MK_F_SILU;
  const int K = st.k, k8 = K / 8;
  const int n_out = silu ? st.n / 2 : st.n;
  const int ntiles = (n_out + 15) / 16;  // output tiles of 16 columns
  const int t_begin = (int)(((long long)c.vid * ntiles) / c.G), t_end = (int)(((long long)(c.vid + 1) * ntiles) / c.G);
  const uint16_t *x = (st.flags & MK_F_NORM) ? (const uint16_t *)st.norm_out : (const uint16_t *)st.in;
  const int ldx = (st.flags & MK_F_NORM) ? st.ld_norm : st.ld_in;
  const bool pipe = (K & 255) == 0;  // every wavefront's K slice is a whole number of 64-wide steps
  const int lgw = pipe ? 16 : 8;     // k elements a lane group owns per step
  const int kq = ((K / 32 + MK_WAVES - 1) / MK_WAVES) * 32;  // K slice per wavefront, multiple of 32
  const int kbeg = min(K, wave * kq), kend = min(K, kbeg + kq);
  const int half = st.silu_half;
  const int otg = silu ? TG / 2 : TG;  // output tiles per sweep
  f32x4 *red = (f32x4 *)smem;           // [waves][TG][MT][64]
  // With a tile-ordered weight copy the step's two operands hold k = 64 s + 8 lg .. and 64 s + 32 + 8 lg .. (the copy's
  // order) and a tile streams contiguously; read from the row-major weights they are the 32 contiguous bytes at
  // k = 64 s + 16 lg.  The token rows follow the same order.
  const bool packed = pipe && st.wpack != nullptr;
  const int wstep = packed ? 128 : 8, whalf = packed ? 64 : 1;  // 16-byte operands between steps / between the halves
  const int xhalf = packed ? 32 : 8;                           // elements between the halves of a token-row step
  const auto xrows = dev_rows(x);
  int xrow[MT];  // bytes
#pragma unroll
  for (int mt = 0; mt < MT; mt++) xrow[mt] = (min(mt * 16 + lr, M - 1) * ldx + (packed ? lg * 8 : lg * lgw)) * 2;

  for (int ot0 = t_begin; ot0 < t_end; ot0 += otg) {
    const int not_ = min(otg, t_end - ot0);       // output tiles in this sweep
    const int nt = silu ? 2 * not_ : not_;        // weight tiles in this sweep
    const uint16_t *wrow[TG];
#pragma unroll
    for (int t = 0; t < TG; t++) {
      const int ot = ot0 + (silu ? (t >> 1) : t);
      int o = min(ot * 16 + lr, n_out - 1);       // output column owned by this lane's weight row
      int vr = o;
      if (silu) {
        const int g = o / half;
        vr = g * 2 * half + (o - g * half) + ((t & 1) ? half : 0);
      }
      wrow[t] = packed ? (const uint16_t *)((const u32x4 *)st.wpack + (size_t)(silu ? 2 * ot + (t & 1) : ot) * (K >> 6) * 128 + lane)
                       : (const uint16_t *)weight_row(st.w, vr, k8) + lg * lgw;
    }
    f32x4 acc[TG][MT];
#pragma unroll
    for (int t = 0; t < TG; t++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) acc[t][mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (pipe) {
      // 64 k per step: a lane owns 32 contiguous bytes of its weight row and of its token row (two matrix-core
      // operands), so the four lane groups of a row cover one whole 128-byte line; NB steps are kept in flight.
      const int nsteps = (kend - kbeg) >> 6;
      bf16x8 a[NB][TG][2], b[NB][MT][2];
      auto load_step = [&](int s_, bf16x8 (&aa)[TG][2], bf16x8 (&bb)[MT][2]) {
        const int k = kbeg + (s_ << 6);
#pragma unroll
        for (int t = 0; t < TG; t++)
          if (t < nt) {
            const bf16x8 *wp = (const bf16x8 *)wrow[t] + (k >> 6) * wstep;
            aa[t][0] = __builtin_nontemporal_load(wp);
            aa[t][1] = __builtin_nontemporal_load(wp + whalf);
          }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
          bb[mt][0] = __builtin_bit_cast(bf16x8, ldc_16B(xrows, xrow[mt] + 2 * k));
          bb[mt][1] = __builtin_bit_cast(bf16x8, ldc_16B(xrows, xrow[mt] + 2 * (k + xhalf)));
        }
      };
#pragma unroll
      for (int j = 0; j < NB; j++)
        if (j < nsteps) load_step(j, a[j], b[j]);
      for (int s0 = 0; s0 < nsteps; s0 += NB) {
#pragma unroll
        for (int j = 0; j < NB; j++) {
          if (s0 + j < nsteps) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
              for (int t = 0; t < TG; t++)
                if (t < nt) {
#pragma unroll
                  for (int mt = 0; mt < MT; mt++) acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j][t][h], b[j][mt][h], acc[t][mt], 0, 0, 0);
                }
            if (s0 + j + NB < nsteps) load_step(s0 + j + NB, a[j], b[j]);
          }
        }
      }
    } else {
#pragma unroll 2
      for (int k = kbeg; k < kend; k += 32) {
        bf16x8 a[TG], b[MT];
#pragma unroll
        for (int t = 0; t < TG; t++)
          if (t < nt) a[t] = __builtin_nontemporal_load((const bf16x8 *)(wrow[t] + k));
#pragma unroll
        for (int mt = 0; mt < MT; mt++) b[mt] = __builtin_bit_cast(bf16x8, ldc_16B(xrows, xrow[mt] + 2 * k));
#pragma unroll
        for (int t = 0; t < TG; t++)
          if (t < nt) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b[mt], acc[t][mt], 0, 0, 0);
          }
      }
    }
    MK_MARK(c, 1);
    __syncthreads();  // previous sweep's epilogue has finished reading LDS
#pragma unroll
    for (int t = 0; t < TG; t++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) red[((wave * TG + t) * MT + mt) * 64 + lane] = acc[t][mt];
    __syncthreads();
    MK_MARK(c, 2);
    // epilogue: entry (output tile u, token tile mt, lane slot l) -> 4 consecutive output columns of one token row
    const int entries = not_ * MT * 64;
    for (int e = tid; e < entries; e += MK_THREADS) {
      const int l = e & 63, mt = (e >> 6) % MT, u = (e >> 6) / MT;
      const int m = mt * 16 + (l & 15);
      const int n0 = (ot0 + u) * 16 + (l >> 4) * 4;
      f32x4 v, v2;
      if (silu) {
        v = red[((0 * TG + 2 * u) * MT + mt) * 64 + l];
        v2 = red[((0 * TG + 2 * u + 1) * MT + mt) * 64 + l];
#pragma unroll
        for (int w = 1; w < MK_WAVES; w++) {
          v += red[((w * TG + 2 * u) * MT + mt) * 64 + l];
          v2 += red[((w * TG + 2 * u + 1) * MT + mt) * 64 + l];
        }
      } else {
        v = red[((0 * TG + u) * MT + mt) * 64 + l];
#pragma unroll
        for (int w = 1; w < MK_WAVES; w++) v += red[((w * TG + u) * MT + mt) * 64 + l];
      }
      if (m < M) {
        uint16_t *orow = (uint16_t *)st.out + (size_t)m * st.ld_out;
        const uint16_t *rrow = (const uint16_t *)st.res + (size_t)m * st.ld_res;
        float rr[4], res[4];
        if (st.flags & MK_F_RES) ldc_bf16x4(rrow, n0, n_out, res);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float r = silu ? linear_glu(st, v[i], v2[i]) : v[i];
          if (st.flags & MK_F_RES) r += res[i];
          rr[i] = linear_act(st, r);
        }
        stc_bf16x4(orow, n0, n_out, rr);
      }
    }
  }
}

// Standalone SwiGLU over interleaved [gate ; up] groups (used when the graph keeps the
// gate/up linear and the activation apart).  Reference task: tasks/mi300/silu_mul_mi300.cuh:42-184.
__device__ __forceinline__ void stage_silu_mul(CStage &st, Ctx &c, int M) {
  barrier_wait(c);
  const int n = st.n, half = st.silu_half;
  const uint16_t *in = (const uint16_t *)st.in;
  uint16_t *out = (uint16_t *)st.out;
  const int total = M * (st.topk > 0 ? st.topk : 1) * n;  // MoE: topk rows per token, contiguous
  for (int i = c.vid * MK_THREADS + c.tid; i < total; i += c.G * MK_THREADS) {
    const int t = i / n, j = i - t * n;
    const int g = j / half, jj = j - g * half;
    const uint16_t *row = in + (size_t)t * st.ld_in + (size_t)g * 2 * half;
    out[(size_t)t * st.ld_out + j] = (uint16_t)f2bf(silu_mul(bf2f(ldc_u16(row + jj)), bf2f(ldc_u16(row + half + jj))));
  }
}

// Row copy.  Reference task: identity_task_impl (tasks/ampere/identity.cuh:24-37).
__device__ __forceinline__ void stage_copy(CStage &st, Ctx &c, int M) {
  barrier_wait(c);
  const uint16_t *in = (const uint16_t *)st.in;
  uint16_t *out = (uint16_t *)st.out;
  const long long total = (long long)M * st.n;
  for (long long i = (long long)c.vid * MK_THREADS + c.tid; i < total; i += (long long)c.G * MK_THREADS) stc_u16(out + i, ldc_u16(in + i));
  c.wrote_through = true;
}

// ----------------------------------------------------------------------------- mixture of experts
// Routing lists of one workgroup, kept in the LDS region above MK_MOE_OFFSET.
struct MoeLds {
  int r[MK_MOE_MAX_EXPERTS];          // single-token routing: 1 + slot per expert
  int act_e[MK_MOE_MAX_EXPERTS];      // expert id of each active expert
  int pair_off[MK_MOE_MAX_EXPERTS + 4];  // first (token, slot) pair of each active expert; [n_act] = number of pairs
  int pair_ts[MK_MAX_TOKENS * MK_MOE_MAX_TOPK];  // token | slot << 8
  int n_act;
  int wtot[2][MK_WAVES];
  float w[MK_MOE_MAX_TOPK];           // single-token routing weights by slot
};

__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp_f32<0x128>(v));
  v = fmaxf(v, dpp_f32<0x124>(v));
  v = fmaxf(v, dpp_f32<0x122>(v));
  v = fmaxf(v, dpp_f32<0x121>(v));
  return fmaxf(fmaxf(lane_f32(v, 0), lane_f32(v, 16)), fmaxf(lane_f32(v, 32), lane_f32(v, 48)));
}

// Arg-max of (value, index) pairs over the wavefront; equal values go to the lower index.  Every lane returns the winner.
__device__ __forceinline__ void group16_argmax(float &bv, int &be) {
#define MK_ARGMAX_STEP(CTRL)                                                 \
  {                                                                          \
    const float ov = dpp_f32<CTRL>(bv);                                      \
    const int oe = __builtin_amdgcn_update_dpp(0, be, CTRL, 0xF, 0xF, true); \
    if (ov > bv || (ov == bv && oe < be)) {                                  \
      bv = ov;                                                               \
      be = oe;                                                               \
    }                                                                        \
  }
  MK_ARGMAX_STEP(0x128)
  MK_ARGMAX_STEP(0x124)
  MK_ARGMAX_STEP(0x122)
  MK_ARGMAX_STEP(0x121)
#undef MK_ARGMAX_STEP
}
__device__ __forceinline__ void wave_argmax(float &bv, int &be) {
  group16_argmax(bv, be);
  float rv = lane_f32(bv, 0);
  int re = __builtin_amdgcn_readlane(be, 0);
#pragma unroll
  for (int r = 16; r < 64; r += 16) {
    const float ov = lane_f32(bv, r);
    const int oe = __builtin_amdgcn_readlane(be, r);
    if (ov > rv || (ov == rv && oe < re)) {
      rv = ov;
      re = oe;
    }
  }
  bv = rv;
  be = re;
}

// The largest of a wavefront's 256 values (value q of lane l has index 64 q + l) and its index, the lower one of equal values; in every lane.  Bound by
// the chain of dependent instructions: a maximum without indices and one comparison per value are 40 of them, pairs of value and index carried
// through the reduction were 100 (eight of 128 experts of each of 16 tokens, as a stage: 6.5 -> 4.9 us).  `none`: the index where no value equals the maximum (all of them NaN).
__device__ __forceinline__ void wave_pick(const float (&p)[4], int none, float &bv, int &be) {
  bv = wave_max(fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3])));
  be = none;
#pragma unroll
  for (int q = 3; q >= 0; q--) {
    const unsigned long long has = __ballot(p[q] == bv);
    if (has) be = q * 64 + (int)__ffsll(has) - 1;
  }
}

// Route one token with one wavefront: fp32 softmax over all experts, `topk` rounds of arg-max (equal probabilities
// go to the lower expert id), weights renormalised by the sum of the selected probabilities.  Lane l owns experts
// l, l+64, ...: sel[j] becomes 1 + slot for a selected expert l + 64 j, 0 otherwise; lane s < topk returns the weight
// and expert of slot s.  Reference task: tasks/mi300/moe_topk_softmax_mi300.cuh:100-213.
// PICK: by wave_pick.  Not inside the single-token expert linear: that stage became 1.1 us shorter, but W2 behind it, whose registers are allotted
// together with it, 1.8 longer (a step of qwen3-30b-a3b, 8 layers, 64 times: 30.15 -> 30.7 ms).
template <bool PICK>
__device__ __forceinline__ void moe_route_wave(const uint16_t *logits, int E, int topk, int lane, int sel[4], float &w_slot, int &e_slot) {
  float p[4];
  float mx = -3.0e38f;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int e = j * 64 + lane;
    p[j] = e < E ? bf2f(ldc_u16(logits + e)) : -3.0e38f;
    mx = fmaxf(mx, p[j]);
    sel[j] = 0;
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    p[j] = (j * 64 + lane < E) ? expf(p[j] - mx) : 0.f;
    sum += p[j];
  }
  const float inv = 1.f / wave_sum(sum);
#pragma unroll
  for (int j = 0; j < 4; j++) p[j] = (j * 64 + lane < E) ? p[j] * inv : -1.f;
  float tot = 0.f;
  w_slot = 0.f;
  e_slot = 0;
  for (int s = 0; s < topk; s++) {
    float bv = p[0];
    int be = lane;
    if constexpr (PICK) {
      wave_pick(p, s, bv, be);
    } else {
#pragma unroll
      for (int j = 1; j < 4; j++)
        if (p[j] > bv) {
          bv = p[j];
          be = j * 64 + lane;
        }
      wave_argmax(bv, be);
    }
    tot += bv;
    if (lane == s) {
      w_slot = bv;
      e_slot = be;
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (j * 64 + lane == be) {
        sel[j] = s + 1;
        p[j] = -10000.f;
      }
  }
  w_slot *= 1.f / tot;
}

// Router stage for multi-token iterations: one wavefront per token writes the routing weights and the token's
// column of the routing table.  Columns of tokens that are not part of the iteration are left alone.
__device__ __forceinline__ void stage_moe_topk(CStage &st, Ctx &c, int M) {
  barrier_wait(c);
  const int lane = c.tid & 63, wave = __builtin_amdgcn_readfirstlane(c.tid >> 6);
  const int E = st.num_experts;
  for (int t = c.vid * MK_WAVES + wave; t < M; t += c.G * MK_WAVES) {
    int sel[4];
    float w;
    int e;
    moe_route_wave<true>((const uint16_t *)st.moe_logits + (size_t)t * st.ld_logits, E, st.topk, lane, sel, w, e);
    if (lane < st.topk) __hip_atomic_store(st.moe_topk_w + (size_t)t * st.ld_topk_w + lane, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (j * 64 + lane < E) __hip_atomic_store(st.moe_routing + (size_t)(j * 64 + lane) * st.ld_routing + t, sel[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  c.wrote_through = true;  // written through: no L2 write-back at this stage's arrival
}

// Build the active-expert list and the (token, slot) pairs of every active expert from the routing table.
// Single-token iterations keep slot order (active expert s is the expert of slot s); multi-token iterations list
// experts in ascending id with their tokens in ascending order.
__device__ __forceinline__ void moe_build_lists(CStage &st, const Ctx &c, MoeLds *L, int M, bool r_in_lds) {
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int E = st.num_experts;
  if (M == 1) {
    if (tid <= st.topk) {  // slot s is "active expert" s; a slot no expert claims (caller-written table) stays empty
      L->act_e[tid] = -1;
      L->pair_off[tid] = tid;
      L->pair_ts[tid] = tid << 8;
    }
    if (tid == 0) L->n_act = st.topk;
    __syncthreads();
    if (tid < E) {
      const int r = r_in_lds ? L->r[tid] : ldc_i32(st.moe_routing + (size_t)tid * st.ld_routing);
      if (r > 0 && r <= st.topk) L->act_e[r - 1] = tid;
    }
    __syncthreads();
    return;
  }
  // the expert's row of the routing table, all requested at once
  int rv[MK_MAX_TOKENS];
  int cnt = 0;
  if (tid < E) {
#pragma unroll
    for (int t = 0; t < MK_MAX_TOKENS; t++)
      if (t < M) rv[t] = ldc_i32(st.moe_routing + (size_t)tid * st.ld_routing + t);
#pragma unroll
    for (int t = 0; t < MK_MAX_TOKENS; t++)
      if (t < M) cnt += rv[t] > 0 && rv[t] <= st.topk;
  }
  int sc = cnt, sa = cnt > 0;  // inclusive scans inside the wavefront
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int vc = __shfl_up(sc, o, 64), va = __shfl_up(sa, o, 64);
    if (lane >= o) {
      sc += vc;
      sa += va;
    }
  }
  if (lane == 63) {
    L->wtot[0][wave] = sc;
    L->wtot[1][wave] = sa;
  }
  __syncthreads();
  int bc = 0, ba = 0;
  for (int w = 0; w < wave; w++) {
    bc += L->wtot[0][w];
    ba += L->wtot[1][w];
  }
  const int off = bc + sc - cnt, ai = ba + sa - (cnt > 0);
  if (cnt > 0) {
    L->act_e[ai] = tid;
    L->pair_off[ai] = off;
    int i = off;
#pragma unroll
    for (int t = 0; t < MK_MAX_TOKENS; t++)
      if (t < M) {
        const int r = rv[t];
        if (r > 0 && r <= st.topk && i < MK_MAX_TOKENS * MK_MOE_MAX_TOPK) L->pair_ts[i++] = t | ((r - 1) << 8);
      }
  }
  if (tid == MK_THREADS - 1) {
    L->n_act = ba + sa;
    L->pair_off[ba + sa] = bc + sc;
  }
  __syncthreads();
}

// Per-expert linear over the active experts of one token, whatever the sizes: y[slot, :] = W[e(slot)] x(slot), one weight row (or one
// [gate ; up] row pair) per wavefront step.  (M is 1.  Written without it and without the token index, the register allocation of the multi-token
// linears in the same kernel moved: a prompt of qwen3-8b 39.7 -> 39.8 ms, with the rule of attn_in_pairs up to 40.4.)
// Work units (active expert, row) are dealt out in contiguous runs per wavefront; the rows of the next R units are
// in flight in registers while a unit is reduced.  Optional epilogues: SwiGLU (gate and up rounded to bf16 first, as
// the separate activation task of the reference sees them) and the weighted sum over the
// slots plus residual, accumulated in slot order in fp32 from the bf16-rounded expert outputs.
// KL = 16-byte row segments per lane (K <= 512 KL).
// Reference tasks: moe_linear_kernel_mi300 (tasks/mi300/moe_linear_mi300.cuh:53-295), silu_mul_task_impl,
// mul_sum_add_mi300_task_impl (tasks/mi300/moe_mul_sum_add_mi300.cuh:31-55).
template <int KL, int R, bool SILU>
__device__ __forceinline__ void stage_moe_linear_t(CStage &st, Ctx &c, int M, char *smem) {
  constexpr int NROW = SILU ? 2 : 1;
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  MoeLds *L = (MoeLds *)(smem + MK_MOE_OFFSET);
  const int k8 = st.k / 8;
  const bool combine = !SILU && (st.flags & MK_F_MOE_COMBINE) && M == 1;
  const bool inline_topk = (st.flags & MK_F_MOE_INLINE_TOPK) && M == 1;
  barrier_wait(c);
  if (inline_topk) {
    if (wave == 0) {
      int sel[4];
      float w;
      int e;
      moe_route_wave<false>((const uint16_t *)st.moe_logits, st.num_experts, st.topk, lane, sel, w, e);
#pragma unroll
      for (int j = 0; j < 4; j++)
        if (j * 64 + lane < st.num_experts) {
          L->r[j * 64 + lane] = sel[j];
          if (c.vid == 0) st.moe_routing[(size_t)(j * 64 + lane) * st.ld_routing] = sel[j];
        }
      if (lane < st.topk) {
        L->w[lane] = w;
        if (c.vid == 0) st.moe_topk_w[lane] = w;
      }
    }
    __syncthreads();
  } else if (combine && tid < st.topk) {
    L->w[tid] = ldc_f32(st.moe_topk_w + tid);
  }
  moe_build_lists(st, c, L, M, inline_topk);
  const int n_act = L->n_act;
  if (c.vid == 0 && st.moe_mask) {  // publish the active-expert list (its order is unspecified in the reference)
    for (int i = tid; i < st.num_experts; i += MK_THREADS) st.moe_mask[i] = i < n_act ? L->act_e[i] : -1;
    if (tid == 0) st.moe_mask[st.num_experts] = n_act;
  }
  // single token: stage the input row(s) in LDS (one row, or one row per slot)
  const int nslot_in = st.ld_in_slot ? st.topk : 1;
  const bool x_lds = M == 1 && (size_t)nslot_in * st.k * 2 <= (size_t)MK_RED_OFFSET;
  u32x4 *xs4 = (u32x4 *)smem;
  if (x_lds) {
    for (int i = tid; i < nslot_in * k8; i += MK_THREADS) {
      const int s = i / k8, o = i - s * k8;
      xs4[i] = ldc_16B((const u32x4 *)((const uint16_t *)st.in + (size_t)s * st.ld_in_slot) + o);
    }
    __syncthreads();
  }
  const int NR = SILU ? st.n / 2 : st.n;  // units per expert
  const int nwaves = c.G * MK_WAVES, gw = c.vid * MK_WAVES + wave;
  int U, upw;
  if (combine) {  // token-major: the n_act units of one output row are consecutive and stay in one wavefront
    U = NR * n_act;
    upw = ((NR + nwaves - 1) / nwaves) * n_act;
  } else {
    U = n_act * NR;
    upw = (U + nwaves - 1) / nwaves;
  }
  const int u0 = min(U, gw * upw), u1 = min(U, u0 + upw);
  const u32x4 *W = (const u32x4 *)st.w.seg[0];
  const u32x4 zero = {0u, 0u, 0u, 0u};
  u32x4 buf[R][NROW][KL];
  auto load_unit = [&](int u, u32x4 (&b)[NROW][KL]) {
    int a, j;
    if (combine) {
      j = u / n_act;
      a = u - j * n_act;
    } else {
      a = u / NR;
      j = u - a * NR;
    }
    const int ei = L->act_e[a];
    const size_t e = (size_t)max(ei, 0);
#pragma unroll
    for (int h = 0; h < NROW; h++) {
      const u32x4 *p = W + (e * st.n + (size_t)(j + h * NR)) * k8;
#pragma unroll
      for (int kc = 0; kc < KL; kc++) b[h][kc] = (ei >= 0 && kc * 64 + lane < k8) ? ldg_stream(p + kc * 64 + lane) : zero;
    }
  };
#pragma unroll
  for (int jj = 0; jj < R; jj++)
    if (u0 + jj < u1) load_unit(u0 + jj, buf[jj]);
  uint16_t *out = (uint16_t *)st.out, *out2 = (uint16_t *)st.out2;
  float comb = 0.f;
  for (int i = u0; i < u1; i += R) {
#pragma unroll
    for (int jj = 0; jj < R; jj++) {
      const int u = i + jj;
      if (u < u1) {
        int a, j;
        if (combine) {
          j = u / n_act;
          a = u - j * n_act;
        } else {
          a = u / NR;
          j = u - a * NR;
        }
        const int p0 = L->pair_off[a], p1 = L->act_e[a] >= 0 ? L->pair_off[a + 1] : p0;
        if (combine && a == 0) comb = bf2f(ldc_u16((const uint16_t *)st.res + j));
        for (int p = p0; p < p1; p++) {
          const int ts = L->pair_ts[p], tok = ts & 255, slot = ts >> 8;
          const u32x4 *x = x_lds ? xs4 + (st.ld_in_slot ? slot * k8 : 0)
                                 : (const u32x4 *)((const uint16_t *)st.in + (size_t)tok * st.ld_in + (size_t)slot * st.ld_in_slot);
          float acc[NROW];
#pragma unroll
          for (int h = 0; h < NROW; h++) acc[h] = 0.f;
#pragma unroll
          for (int kc = 0; kc < KL; kc++) {
            u32x4 xv = zero;
            if (kc * 64 + lane < k8) xv = x_lds ? x[kc * 64 + lane] : ldc_16B(x + kc * 64 + lane);
#pragma unroll
            for (int h = 0; h < NROW; h++) acc[h] = dot8(buf[jj][h][kc], xv, acc[h]);
          }
#pragma unroll
          for (int h = 0; h < NROW; h++) acc[h] = wave_sum(acc[h]);
          uint16_t *y = out + (size_t)tok * st.ld_out + (size_t)slot * st.ld_out_slot;
          if (SILU) {
            const uint32_t g = f2bf(acc[0]), up = f2bf(acc[NROW - 1]);
            if (lane == 0) {
              y[j] = (uint16_t)g;
              y[j + NR] = (uint16_t)up;
              out2[(size_t)tok * st.ld_out2 + (size_t)slot * st.ld_out2_slot + j] = (uint16_t)f2bf(silu_mul(bf2f((uint16_t)g), bf2f((uint16_t)up)));
            }
          } else {
            const uint32_t v = f2bf(acc[0]);
            if (lane == 0) y[j] = (uint16_t)v;
            if (combine) comb = fmaf(bf2f((uint16_t)v), L->w[slot], comb);
          }
        }
        if (combine && a == n_act - 1 && lane == 0) out2[j] = (uint16_t)f2bf(comb);
        if (u + R < u1) load_unit(u + R, buf[jj]);
      }
    }
  }
}

// Single-token per-expert linear, tuned like the dense single-token linear: wavefront 0 polls the barrier, routes
// (or reads the routing of the stage before), stages the input row(s) and publishes the routing outputs; wavefronts
// 1..3 draw work from the workgroup's LDS ticket counter with R tickets of weight rows in flight each.  A ticket is
// one [gate ; up] row pair of one slot's expert (SILU) or, for the W2 + weighted-sum form, output row j of ALL TK
// slots' experts, so the combine stays inside one wavefront.  When the stage directly before was the W13 stage of the
// same token its expert list is still in LDS: the first tickets' rows are then requested before the barrier.  All
// outputs are written through.
template <int KL, int R, bool SILU>
__device__ __forceinline__ void stage_moe_linear_m1(CStage &st, Ctx &c, char *smem) {
  constexpr int TK = 8;
  constexpr int NSUB = SILU ? 2 : TK;
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  MoeLds *L = (MoeLds *)(smem + MK_MOE_OFFSET);
  const int k8 = st.k / 8, topk = st.topk, E = st.num_experts;
  const bool ctrl = wave == 0;
  const bool inline_topk = st.flags & MK_F_MOE_INLINE_TOPK;
  const int NR = SILU ? st.n / 2 : st.n;
  const int n_tk = SILU ? topk * NR : NR;
  const int tq = n_tk / c.G, trem = n_tk - tq * c.G;
  const int t_begin = c.vid * tq + min(c.vid, trem), t_end = t_begin + tq + (c.vid < trem ? 1 : 0);
  int *ticket = c.sh_ticket + (c.seq & 1);
  const bool reuse = !inline_topk && __builtin_amdgcn_readfirstlane(c.sh_ticket[2]) == c.seq - 1;
  const u32x4 *W = (const u32x4 *)st.w.seg[0];
  u32x4 *xs4 = (u32x4 *)smem;
  const u32x4 zero = {0u, 0u, 0u, 0u};
  auto take = [&]() -> int {
    int t = 0;
    if (lane == 0) t = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    t = __builtin_amdgcn_readfirstlane(t) + t_begin;
    return t < t_end ? t : -1;
  };
  // W2 form: the weight base of every slot's expert, fixed for the whole stage (set once the expert list is known)
  const u32x4 *eb[SILU ? 1 : TK];
  bool ev[SILU ? 1 : TK];
  auto set_bases = [&]() {
    if (!SILU) {
#pragma unroll
      for (int h = 0; h < (SILU ? 1 : TK); h++) {
        const int ei = __builtin_amdgcn_readfirstlane(L->act_e[h]);
        ev[h] = ei >= 0;
        eb[h] = W + (size_t)max(ei, 0) * st.n * k8 + lane;
      }
    }
  };
  auto load_ticket = [&](int tk, u32x4 (&b)[NSUB][KL]) {
    if (SILU) {
      const int a = tk / NR, j = tk - a * NR;
      const int ei = __builtin_amdgcn_readfirstlane(L->act_e[a]);
#pragma unroll
      for (int h = 0; h < NSUB; h++) {
        const u32x4 *p = W + ((size_t)max(ei, 0) * st.n + (size_t)(j + h * NR)) * k8;
#pragma unroll
        for (int kc = 0; kc < KL; kc++) b[h][kc] = (ei >= 0 && kc * 64 + lane < k8) ? ldg_stream(p + kc * 64 + lane) : zero;
      }
    } else {
#pragma unroll
      for (int h = 0; h < NSUB; h++) {
        const u32x4 *p = eb[SILU ? 0 : h] + (size_t)tk * k8;
#pragma unroll
        for (int kc = 0; kc < KL; kc++) b[h][kc] = (ev[SILU ? 0 : h] && kc * 64 + lane < k8) ? ldg_stream(p + kc * 64) : zero;
      }
    }
  };
  u32x4 buf[R][NSUB][KL];
  int ut[R];
#pragma unroll
  for (int j = 0; j < R; j++) ut[j] = -1;
  // W2 form after the W13 stage of the same token: the experts are known before the barrier, and a workgroup's whole
  // share of the weights (a few tickets of TK rows) fits the idle LDS above the routing lists.  Each worker wavefront
  // keeps its R tickets in flight as a rolling window: a ticket that has landed is parked in LDS and its slot refilled,
  // NLP tickets per wavefront; they are reduced from LDS once the input rows are there.
  constexpr int NLP = SILU ? 0 : MK_TUNE_MOE_M1_PARK;
  constexpr int PARK_OFF = MK_MOE_OFFSET + 8192;
  static_assert(sizeof(MoeLds) <= 8192, "routing lists overlap the parked rows");
  static_assert(PARK_OFF + (MK_WAVES - 1) * NLP * NSUB * KL * 1024 <= MK_LDS_BYTES, "parked rows exceed the LDS window");
  u32x4 *lrows = (u32x4 *)(smem + PARK_OFF) + (size_t)(wave > 0 ? wave - 1 : 0) * (NLP > 0 ? NLP : 1) * NSUB * KL * 64;
  int lo_[NLP > 0 ? NLP : 1];
#pragma unroll
  for (int i = 0; i < (NLP > 0 ? NLP : 1); i++) lo_[i] = -1;
  if (!ctrl) {
    if (reuse) {
      set_bases();
#pragma unroll
      for (int i = 0; i < NLP + R; i++) {
        const int sl = i % R;
        if (i >= R) {
#pragma unroll
          for (int h = 0; h < NSUB; h++)
#pragma unroll
            for (int kc = 0; kc < KL; kc++) lrows[(((i - R) * NSUB + h) * KL + kc) * 64 + lane] = buf[sl][h][kc];
          lo_[i - R] = ut[sl];
        }
        ut[sl] = take();
        if (ut[sl] >= 0) load_ticket(ut[sl], buf[sl]);
      }
    }
  } else {
    if (c.pending && tid == 0) barrier_poll(c);
    // input row(s): one row, or one row per slot (at most 12 16-byte segments per lane)
    const int nx = (st.ld_in_slot ? topk : 1) * k8;
    u32x4 xv[12];
#pragma unroll
    for (int i = 0; i < 12; i++) {
      const int ci = i * 64 + lane;
      if (ci < nx) {
        const int sl = ci / k8, o = ci - sl * k8;
        xv[i] = ldc_16B((const u32x4 *)((const uint16_t *)st.in + (size_t)sl * st.ld_in_slot) + o);
      }
    }
    if (inline_topk) {
      int sel[4];
      float w;
      int e;
      moe_route_wave<false>((const uint16_t *)st.moe_logits, E, topk, lane, sel, w, e);
      if (lane < topk) {
        L->act_e[lane] = e;
        L->w[lane] = w;
        if (c.vid == 0) __hip_atomic_store(st.moe_topk_w + lane, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      if (c.vid == 0) {
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (j * 64 + lane < E) __hip_atomic_store(st.moe_routing + (size_t)(j * 64 + lane) * st.ld_routing, sel[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    } else if (!reuse) {
      if (lane < topk) L->act_e[lane] = -1;
#pragma unroll
      for (int j = 0; j < 4; j++)
        if (j * 64 + lane < E) {
          const int r = ldc_i32(st.moe_routing + (size_t)(j * 64 + lane) * st.ld_routing);
          if (r > 0 && r <= topk) L->act_e[r - 1] = j * 64 + lane;
        }
      if (!SILU && lane < topk) L->w[lane] = ldc_f32(st.moe_topk_w + lane);
    }
#pragma unroll
    for (int i = 0; i < 12; i++)
      if (i * 64 + lane < nx) xs4[i * 64 + lane] = xv[i];
    if (lane == 0) c.sh_ticket[2] = c.seq;
  }
  __syncthreads();
  barrier_done(c);
  // outputs are collected in LDS ([array][ticket - t_begin]) and written out together once every worker is done
  uint16_t *so = (uint16_t *)(smem + MK_OUT_OFFSET);
  const int n_loc = t_end - t_begin;
  constexpr int NARR = SILU ? 3 : TK + 1;
  auto flush = [&]() {
    __syncthreads();
    uint16_t *o1 = (uint16_t *)st.out, *o2 = (uint16_t *)st.out2;
    for (int i = tid; i < NARR * n_loc; i += MK_THREADS) {
      const int arr = i / n_loc, tk = t_begin + (i - arr * n_loc);
      uint16_t *dst;
      if (SILU) {
        const int a = tk / NR, row = tk - a * NR;
        dst = arr == 2 ? o2 + (size_t)a * st.ld_out2_slot + row : o1 + (size_t)a * st.ld_out_slot + row + arr * NR;
      } else {
        if (arr < TK && L->act_e[arr] < 0) continue;
        dst = arr == TK ? o2 + tk : o1 + (size_t)arr * st.ld_out_slot + tk;
      }
      stc_u16(dst, so[i]);
    }
    c.wrote_through = true;
  };
  if (ctrl) {
    if (c.vid == 0 && st.moe_mask) {  // active-expert list (its order is unspecified in the reference) and count
      for (int i = lane; i < E; i += 64) __hip_atomic_store(st.moe_mask + i, i < topk ? L->act_e[i] : -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (lane == 0) __hip_atomic_store(st.moe_mask + E, topk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (!reuse || ctrl) set_bases();
  // the staged input row(s) stay in registers for the whole stage
  u32x4 xr[SILU ? 1 : TK][KL];
#pragma unroll
  for (int h = 0; h < (SILU ? 1 : TK); h++)
#pragma unroll
    for (int kc = 0; kc < KL; kc++) xr[h][kc] = (kc * 64 + lane < k8) ? xs4[(st.ld_in_slot ? h * k8 : 0) + kc * 64 + lane] : zero;
  float ures[R];
#pragma unroll
  for (int j = 0; j < R; j++) {
    if (!reuse || ctrl) {  // the control wavefront joins the streaming once its part is done
      ut[j] = take();
      if (ut[j] >= 0) load_ticket(ut[j], buf[j]);
    }
    ures[j] = (!SILU && ut[j] >= 0) ? bf2f(ldc_u16((const uint16_t *)st.res + ut[j])) : 0.f;
  }
  if constexpr (NLP > 0) {
    // the parked tickets first: no memory traffic, the register slots keep landing meanwhile
    float lres[NLP];
#pragma unroll
    for (int i = 0; i < NLP; i++) lres[i] = lo_[i] >= 0 ? bf2f(ldc_u16((const uint16_t *)st.res + lo_[i])) : 0.f;
#pragma unroll
    for (int i = 0; i < NLP; i++) {
      if (lo_[i] >= 0) {
        const int tk = lo_[i];
        float acc[NSUB];
#pragma unroll
        for (int h = 0; h < NSUB; h++) {
          acc[h] = 0.f;
#pragma unroll
          for (int kc = 0; kc < KL; kc++) acc[h] = dot8(lrows[((i * NSUB + h) * KL + kc) * 64 + lane], xr[SILU ? 0 : h][kc], acc[h]);
        }
#pragma unroll
        for (int h = 0; h < NSUB; h++) acc[h] = wave_sum(acc[h]);
        float comb = lres[i];
#pragma unroll
        for (int h = 0; h < NSUB; h++) {
          const uint32_t v = f2bf(acc[h]);
          if (lane == 0) so[h * n_loc + tk - t_begin] = (uint16_t)v;
          comb = fmaf(bf2f((uint16_t)v), L->w[SILU ? 0 : h], comb);
        }
        if (lane == 0) so[TK * n_loc + tk - t_begin] = (uint16_t)f2bf(comb);
      }
    }
  }
  while (true) {
    bool any = false;
#pragma unroll
    for (int j = 0; j < R; j++) {
      if (ut[j] >= 0) {
        any = true;
        const int tk = ut[j];
        int a = 0, row = tk;
        if (SILU) {
          a = tk / NR;
          row = tk - a * NR;
        }
        float acc[NSUB];
#pragma unroll
        for (int h = 0; h < NSUB; h++) {
          acc[h] = 0.f;
#pragma unroll
          for (int kc = 0; kc < KL; kc++) {
            acc[h] = dot8(buf[j][h][kc], xr[SILU ? 0 : h][kc], acc[h]);
          }
        }
        const float r0 = ures[j];
        ut[j] = take();
        if (ut[j] >= 0) {
          load_ticket(ut[j], buf[j]);
          if (!SILU) ures[j] = bf2f(ldc_u16((const uint16_t *)st.res + ut[j]));
        }
#pragma unroll
        for (int h = 0; h < NSUB; h++) acc[h] = wave_sum(acc[h]);
        if (SILU) {
          const uint32_t g = f2bf(acc[0]), up = f2bf(acc[1]);
          if (lane == 0) {
            so[tk - t_begin] = (uint16_t)g;
            so[n_loc + tk - t_begin] = (uint16_t)up;
            so[2 * n_loc + tk - t_begin] = (uint16_t)f2bf(silu_mul(bf2f((uint16_t)g), bf2f((uint16_t)up)));
          }
        } else {
          float comb = r0;
#pragma unroll
          for (int h = 0; h < NSUB; h++) {
            const uint32_t v = f2bf(acc[h]);
            if (lane == 0) so[h * n_loc + tk - t_begin] = (uint16_t)v;
            comb = fmaf(bf2f((uint16_t)v), L->w[h], comb);
          }
          if (lane == 0) so[TK * n_loc + tk - t_begin] = (uint16_t)f2bf(comb);
        }
      }
    }
    if (!any) break;
  }
  flush();
}

// Multi-token per-expert linear.  Work units (active expert, row) in expert-major order are split over the workgroups
// by cost (a workgroup then touches one or two experts) and drawn from the LDS ticket counter by all four wavefronts.
// The input rows of the tokens routed to the workgroup's experts are staged in LDS once and the outputs are collected
// in an LDS tile, so the loop over an expert's tokens contains NO vector-memory instruction: the compiler can then
// count the weight-row loads in flight exactly, and R units' rows really stay in flight (with a store inside that
// loop every unit waited for all outstanding loads).  The tile is written out at the end, one contiguous run of
// rows per (token, slot).  A workgroup whose tile or staged rows do not fit runs a plain loop over the same units.
template <int KL, int R, bool SILU>
__device__ __forceinline__ void stage_moe_linear_multi(CStage &st, Ctx &c, int M, bool reuse, char *smem) {
  constexpr int NROW = SILU ? 2 : 1;
  constexpr int NARR = SILU ? 3 : 1;
  const int tid = c.tid, lane = tid & 63;
  MoeLds *L = (MoeLds *)(smem + MK_MOE_OFFSET);
  const int k8 = st.k / 8;
  const int n_act = L->n_act;
  const int NR = SILU ? st.n / 2 : st.n;  // units per expert
  const int n_units = n_act * NR;
  // A unit of expert a costs one row load (RC, in units of one reduction) plus one reduction per token routed to a: split
  // the units so that every workgroup gets the same cost.  With w_a = tokens(a) + RC the cost before expert a is
  // NR * (pair_off[a] + RC * a).
  constexpr int RC = SILU ? MK_TUNE_MOE_ROWCOST13 : MK_TUNE_MOE_ROWCOST2;
  int *bnd = L->wtot[0];  // reused: the scans of the list building are done
  if (tid < 2) bnd[tid] = 0;
  __syncthreads();
  if (tid == 0) c.sh_ticket[2] = ~c.seq;  // (everybody has looked at it)
  const long long total = (long long)NR * (L->pair_off[n_act] + RC * n_act);
  const long long tgt0 = total * c.vid / c.G, tgt1 = total * (c.vid + 1) / c.G;
  if (tid < n_act) {
    const long long before = (long long)NR * (L->pair_off[tid] + RC * tid);
    if (before <= tgt0) __hip_atomic_fetch_max(&bnd[0], tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (before <= tgt1) __hip_atomic_fetch_max(&bnd[1], tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __syncthreads();
  auto unit_at = [&](long long tgt, int a) -> int {
    if (n_act == 0) return 0;
    const long long before = (long long)NR * (L->pair_off[a] + RC * a);
    const int w = L->pair_off[a + 1] - L->pair_off[a] + RC;
    return a * NR + min(NR, (int)((tgt - before) / w));
  };
  const int u_begin = __builtin_amdgcn_readfirstlane(unit_at(tgt0, bnd[0]));
  const int u_end = __builtin_amdgcn_readfirstlane(c.vid == c.G - 1 ? n_units : unit_at(tgt1, bnd[1]));
  const int nu = u_end - u_begin;
  int p_base = 0, n_pairs = 0, maxp = 0;
  if (nu > 0) {
    const int a0 = u_begin / NR, a1 = (u_end - 1) / NR;
    p_base = L->pair_off[a0];
    n_pairs = L->pair_off[a1 + 1] - p_base;
    for (int a = a0; a <= a1; a++) maxp = max(maxp, L->pair_off[a + 1] - L->pair_off[a]);
  }
  // the decision below is per workgroup (uniform within it); either form covers exactly [u_begin, u_end)
  const u32x4 zero = {0u, 0u, 0u, 0u};
  const u32x4 *W = (const u32x4 *)st.w.seg[0];
  const bool plain = (size_t)n_pairs * k8 * 16 > (size_t)(MK_LDS_BYTES - MK_MOE_X_OFFSET) || (size_t)NARR * maxp * nu * 2 > (size_t)MK_MOE_OFFSET;
  int *ticket = c.sh_ticket + (c.seq & 1);
  auto take = [&](int n) -> int {  // first of the next n units of this workgroup (may lie at or beyond u_end)
    int t = 0;
    if (lane == 0) t = __hip_atomic_fetch_add(ticket, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    return __builtin_amdgcn_readfirstlane(t) + u_begin;
  };
  // Every row load is unconditional: a unit at or beyond the end of the range re-reads the range's last unit and is
  // not reduced.  (With the loads under a branch every wait for one unit's rows drained the other units' loads too.)
  auto load_unit = [&](int u_, u32x4 (&b)[NROW][KL]) {
    const int u = min(u_, u_end - 1);
    const int a = u / NR, j = u - a * NR;
    const size_t e = (size_t)__builtin_amdgcn_readfirstlane(L->act_e[a]);
#pragma unroll
    for (int h = 0; h < NROW; h++) {
      const u32x4 *p = W + (e * st.n + (size_t)(j + h * NR)) * k8;
#pragma unroll
      for (int kc = 0; kc < KL; kc++) b[h][kc] = ldg_stream(p + min(kc * 64 + lane, k8 - 1));  // lanes past the row re-read its last segment; their products are dropped below
    }
  };
  // two groups of units in flight: while one is reduced the other one's rows are landing; tickets only grow, so the
  // first group found beyond the range ends the loop
  constexpr int QA = (R + 1) / 2, QB = R / 2;
  u32x4 bufA[QA][NROW][KL], bufB[QB > 0 ? QB : 1][NROW][KL];
  int gA = u_end, gB = u_end;
  auto fill = [&]() {
    gA = take(QA);
#pragma unroll
    for (int q = 0; q < QA; q++) load_unit(gA + q, bufA[q]);
    if (QB > 0) {
      gB = take(QB);
#pragma unroll
      for (int q = 0; q < QB; q++) load_unit(gB + q, bufB[q]);
    }
  };
  // with the lists of the stage before, the first groups' rows are requested before the barrier is awaited (not the polling wavefront's:
  // they would hold up the poll)
  const bool early = !SILU && reuse && nu > 0 && !plain && __builtin_amdgcn_readfirstlane(tid >> 6) != 0;
  if (early) fill();
  if (!SILU && reuse) {
    barrier_wait(c);
  }
  const auto x_rows = dev_rows(st.in);
  if (plain) {
    // too many tokens on this workgroup's experts for the LDS windows: plain form over the same unit range
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint16_t *out = (uint16_t *)st.out, *out2 = (uint16_t *)st.out2;
    for (int u = u_begin + wv; u < u_end; u += MK_WAVES) {
      const int a = u / NR, j = u - a * NR;
      const size_t e = (size_t)L->act_e[a];
      for (int p = L->pair_off[a]; p < L->pair_off[a + 1]; p++) {
        const int ts = L->pair_ts[p], tok = ts & 255, slot = ts >> 8;
        const int x = (tok * st.ld_in + slot * st.ld_in_slot) * 2;  // bytes
        float acc[NROW];
#pragma unroll
        for (int h = 0; h < NROW; h++) {
          acc[h] = 0.f;
          const u32x4 *wr = W + (e * st.n + (size_t)(j + h * NR)) * k8;
          for (int kc = lane; kc < k8; kc += 64) acc[h] = dot8(wr[kc], ldc_16B(x_rows, x + kc * 16), acc[h]);
          acc[h] = wave_sum(acc[h]);
        }
        uint16_t *y = out + (size_t)tok * st.ld_out + (size_t)slot * st.ld_out_slot;
        if (SILU) {
          const uint32_t g = f2bf(acc[0]), up = f2bf(acc[NROW - 1]);
          if (lane == 0) {
            y[j] = (uint16_t)g;
            y[j + NR] = (uint16_t)up;
            out2[(size_t)tok * st.ld_out2 + (size_t)slot * st.ld_out2_slot + j] = (uint16_t)f2bf(silu_mul(bf2f((uint16_t)g), bf2f((uint16_t)up)));
          }
        } else if (lane == 0) {
          y[j] = (uint16_t)f2bf(acc[0]);
        }
      }
    }
    return;
  }
  u32x4 *xs4 = (u32x4 *)(smem + MK_MOE_X_OFFSET);
  uint16_t *so = (uint16_t *)smem;  // [array][pair of the expert][unit - u_begin]
  auto reduce_unit = [&](const u32x4 (&b)[NROW][KL], int u) {
    const int a = u / NR;
    const int p0 = __builtin_amdgcn_readfirstlane(L->pair_off[a]), p1 = __builtin_amdgcn_readfirstlane(L->pair_off[a + 1]);
    for (int p = p0; p < p1; p++) {  // LDS only in here
      const u32x4 *x = xs4 + (p - p_base) * k8;
      float acc[NROW];
#pragma unroll
      for (int h = 0; h < NROW; h++) acc[h] = 0.f;
#pragma unroll
      for (int kc = 0; kc < KL; kc++) {
        const u32x4 xv = (kc * 64 + lane < k8) ? x[kc * 64 + lane] : zero;
#pragma unroll
        for (int h = 0; h < NROW; h++) acc[h] = dot8(b[h][kc], xv, acc[h]);
      }
#pragma unroll
      for (int h = 0; h < NROW; h++) acc[h] = wave_sum(acc[h]);
      uint16_t *t0 = so + (size_t)(p - p0) * nu + (u - u_begin);
      if (SILU) {
        const uint32_t g = f2bf(acc[0]), up = f2bf(acc[NROW - 1]);
        if (lane == 0) {
          t0[0] = (uint16_t)g;
          t0[(size_t)maxp * nu] = (uint16_t)up;
          t0[(size_t)2 * maxp * nu] = (uint16_t)f2bf(silu_mul(bf2f((uint16_t)g), bf2f((uint16_t)up)));
        }
      } else if (lane == 0) {
        t0[0] = (uint16_t)f2bf(acc[0]);
      }
    }
  };
  // The units of a group are consecutive rows, nearly always of one expert: they are then reduced jointly per (token,
  // slot) pair -- the pair's input segments are read from LDS once for all of them and their sums are reduced together
  // (transposing reduction, lane q * NROW + h gets unit q's sum h).  A group that straddles two experts takes the
  // unit-by-unit form.
  auto reduce_group = [&](auto &bufs, int g, auto nqc) {
    constexpr int NQ = decltype(nqc)::value;
    constexpr int NVAL = NQ * NROW;
    constexpr int NV = NVAL <= 1 ? 1 : (NVAL <= 2 ? 2 : (NVAL <= 4 ? 4 : (NVAL <= 8 ? 8 : 16)));
    static_assert(NVAL <= 16, "group size");
    const int nvalid = min(NQ, u_end - g);
    const int a = g / NR;
    if ((g + nvalid - 1) / NR != a) {
#pragma unroll
      for (int q = 0; q < NQ; q++)
        if (q < nvalid) reduce_unit(bufs[q], g + q);
      return;
    }
    const int p0 = __builtin_amdgcn_readfirstlane(L->pair_off[a]), p1 = __builtin_amdgcn_readfirstlane(L->pair_off[a + 1]);
    for (int p = p0; p < p1; p++) {  // LDS only in here
      const u32x4 *x = xs4 + (p - p_base) * k8;
      float vv[NV];
#pragma unroll
      for (int i = 0; i < NV; i++) vv[i] = 0.f;
#pragma unroll
      for (int kc = 0; kc < KL; kc++) {
        const u32x4 xv = (kc * 64 + lane < k8) ? x[kc * 64 + lane] : zero;
#pragma unroll
        for (int q = 0; q < NQ; q++)
#pragma unroll
          for (int h = 0; h < NROW; h++) vv[q * NROW + h] = dot8(bufs[q][h][kc], xv, vv[q * NROW + h]);
      }
      const float tot = transpose_sum<NV>(vv, lane);
      const int q = lane / NROW;
      uint16_t *t0 = so + (size_t)(p - p0) * nu + (g + q - u_begin);
      if (SILU) {
        const float upv = dpp_f32<0x101>(tot);  // row_shl:1: the up sum sits one lane above the gate sum
        const uint32_t gb = f2bf(tot), ub = f2bf(upv);
        if (lane < NVAL && (lane & 1) == 0 && q < nvalid) {
          t0[0] = (uint16_t)gb;
          t0[(size_t)maxp * nu] = (uint16_t)ub;
          t0[(size_t)2 * maxp * nu] = (uint16_t)f2bf(silu_mul(bf2f((uint16_t)gb), bf2f((uint16_t)ub)));
        }
      } else if (lane < NVAL && q < nvalid) {
        t0[0] = (uint16_t)f2bf(tot);
      }
    }
  };
  // stage the input rows of the (token, slot) pairs of this workgroup's experts
  for (int i0 = tid; i0 < n_pairs * k8; i0 += 4 * MK_THREADS) {
    u32x4 v[4];
#pragma unroll
    for (int z = 0; z < 4; z++) {
      const int i = min(i0 + z * MK_THREADS, n_pairs * k8 - 1), p = i / k8, o = i - p * k8;
      const int ts = L->pair_ts[p_base + p], tok = ts & 255, slot = ts >> 8;
      v[z] = ldc_16B(x_rows, (tok * st.ld_in + slot * st.ld_in_slot) * 2 + o * 16);
    }
#pragma unroll
    for (int z = 0; z < 4; z++)
      if (i0 + z * MK_THREADS < n_pairs * k8) xs4[i0 + z * MK_THREADS] = v[z];
  }
  __syncthreads();
  if (nu > 0) {
    if (!early) fill();
    while (gA < u_end) {
      reduce_group(bufA, gA, std::integral_constant<int, QA>{});
      gA = take(QA);
#pragma unroll
      for (int q = 0; q < QA; q++) load_unit(gA + q, bufA[q]);
      if (QB > 0) {
        if (gB >= u_end) break;
        reduce_group(bufB, gB, std::integral_constant<int, (QB > 0 ? QB : 1)>{});
        gB = take(QB);
#pragma unroll
        for (int q = 0; q < QB; q++) load_unit(gB + q, bufB[q]);
      }
    }
  }
  __syncthreads();
  // write the tile out: consecutive threads take consecutive rows of one (token, slot)
  uint16_t *out = (uint16_t *)st.out, *out2 = (uint16_t *)st.out2;
  for (int i = tid; i < NARR * maxp * nu; i += MK_THREADS) {
    const int arr = i / (maxp * nu), r = i - arr * maxp * nu, pi = r / nu, ui = r - pi * nu;
    const int u = u_begin + ui, a = u / NR, j = u - a * NR;
    const int p = L->pair_off[a] + pi;
    if (p >= L->pair_off[a + 1]) continue;
    const int ts = L->pair_ts[p], tok = ts & 255, slot = ts >> 8;
    if (SILU && arr == 2) stc_u16(out2 + (size_t)tok * st.ld_out2 + (size_t)slot * st.ld_out2_slot + j, so[i]);
    else stc_u16(out + (size_t)tok * st.ld_out + (size_t)slot * st.ld_out_slot + j + (arr == 1 ? NR : 0), so[i]);
  }
  c.wrote_through = true;  // (the plain form above returns before this and keeps the write-back)
}

__device__ __forceinline__ void stage_moe_linear(CStage &st, Ctx &c, int M, char *smem) {
  const bool silu = st.flags & MK_F_SILU;
  if (M == 1) {
    // tuned single-token forms: W13 + SwiGLU (one input row), W2 + weighted sum over exactly 8 slots
    const int nx = (st.ld_in_slot ? st.topk : 1) * (st.k / 8);
    const int n_loc = (silu ? st.topk * (st.n / 2) : st.n) / c.G + 1;
    if ((silu ? 3 : 9) * n_loc * 2 > MK_MOE_OFFSET - MK_OUT_OFFSET) {
      // outputs of one workgroup do not fit the LDS collection window: generic form below
    } else if (silu && !st.ld_in_slot && nx <= 768) {
      if (st.k <= 1024) return stage_moe_linear_m1<2, 4, true>(st, c, smem);
      if (st.k <= 2048) return stage_moe_linear_m1<4, MK_TUNE_MOE_M1_R13, true>(st, c, smem);
    } else if (!silu && (st.flags & MK_F_MOE_COMBINE) && st.ld_in_slot && st.topk == 8 && nx <= 768) {
      if (st.k <= 1024) return stage_moe_linear_m1<2, MK_TUNE_MOE_M1_R2, false>(st, c, smem);
    }
  }
  if (M > 1) {
    // common front: wait for the previous stage, routing lists.  Directly behind
    // another expert linear over the same routing table (W2 behind W13) the lists are still in LDS: that stage starts its stream ahead of the
    // barrier.  qwen3-30b-a3b, 16 tokens, W2: 61 -> 51 us.  (Rows of up to 1024 only: in the instances for longer ones, which have no such
    // stage here, it moved the register allocation of the multi-token linears, a prompt of qwen3-8b 50.1 -> 50.7 ms.)
    MoeLds *L = (MoeLds *)(smem + MK_MOE_OFFSET);
    bool reuse = !silu && st.k <= 1024 && __builtin_amdgcn_readfirstlane(c.sh_ticket[2]) == ~(c.seq - 1);
    if (reuse) {
      CStage &pv = (&st)[-1];
      reuse = pv.op == MK_OP_MOE_LINEAR && pv.moe_routing == st.moe_routing && pv.num_experts == st.num_experts && pv.topk == st.topk && pv.ld_routing == st.ld_routing;
    }
    if (!reuse) {
      barrier_wait(c);
      moe_build_lists(st, c, L, M, false);
    }
    if (!(reuse && (&st)[-1].moe_mask == st.moe_mask) && c.vid == 0 && st.moe_mask) {  // publish the active-expert list (its order is unspecified in the reference)
      const int n_act = L->n_act;
      for (int i = c.tid; i < st.num_experts; i += MK_THREADS) st.moe_mask[i] = i < n_act ? L->act_e[i] : -1;
      if (c.tid == 0) st.moe_mask[st.num_experts] = n_act;
    }
    if (st.k <= 1024) {
      if (silu) stage_moe_linear_multi<2, 4, true>(st, c, M, false, smem);
      else stage_moe_linear_multi<2, MK_TUNE_MOE_R2, false>(st, c, M, reuse, smem);
    } else if (st.k <= 2048) {
      if (silu) stage_moe_linear_multi<4, MK_TUNE_MOE_R13, true>(st, c, M, false, smem);
      else stage_moe_linear_multi<4, 4, false>(st, c, M, false, smem);
    } else {
      if (silu) stage_moe_linear_multi<8, 1, true>(st, c, M, false, smem);
      else stage_moe_linear_multi<8, 2, false>(st, c, M, false, smem);
    }
    return;
  }
  if (st.k <= 1024) {
    if (silu) stage_moe_linear_t<2, 4, true>(st, c, M, smem);
    else stage_moe_linear_t<2, 6, false>(st, c, M, smem);
  } else if (st.k <= 2048) {
    if (silu) stage_moe_linear_t<4, 3, true>(st, c, M, smem);
    else stage_moe_linear_t<4, 4, false>(st, c, M, smem);
  } else {
    if (silu) stage_moe_linear_t<8, 1, true>(st, c, M, smem);
    else stage_moe_linear_t<8, 2, false>(st, c, M, smem);
  }
}

// Weighted sum of the expert outputs plus residual for multi-token iterations:
// out[t, :] = bf16(res[t, :] + sum_k w[t, k] * y[t, k, :]), fp32, slots in order.
// Reference task: mul_sum_add_mi300_task_impl (tasks/mi300/moe_mul_sum_add_mi300.cuh:31-55).
__device__ __forceinline__ void stage_moe_combine(CStage &st, Ctx &c, int M) {
  barrier_wait(c);
  const int n = st.n, total = M * n;
  const uint16_t *in = (const uint16_t *)st.in, *res = (const uint16_t *)st.res;
  uint16_t *out = (uint16_t *)st.out;
  for (int i = c.vid * MK_THREADS + c.tid; i < total; i += c.G * MK_THREADS) {
    const int t = i / n, j = i - t * n;
    float s = bf2f(ldc_u16(res + (size_t)t * st.ld_res + j));
    for (int k = 0; k < st.topk; k++)
      s = fmaf(bf2f(ldc_u16(in + (size_t)t * st.ld_in + (size_t)k * st.ld_in_slot + j)), ldc_f32(st.moe_topk_w + (size_t)t * st.ld_topk_w + k), s);
    stc_u16(out + (size_t)t * st.ld_out + j, (uint16_t)f2bf(s));
  }
  c.wrote_through = true;
}

// One 128-wide head row by one wavefront (lane l owns elements l and l + 64, the two halves of a rotation pair): query and key rows
// get the per-head RMSNorm and the rotate-half RoPE, a value row is copied as it is.  The normalised value is rounded to bf16 before
// the rotation, as in the reference (tasks/mi300/kv_cache_update_mi300.cuh:129-182).
struct AttnRow {
  int tok, off, pos;  // row and first column in the q/k/v tensor, position
  int kind;           // 0 query, 1 key, 2 value
  uint16_t *dst;      // LDS
};
// Where these rows come from: stored by the producing linear, or -- when it left its K-slice partials to this stage -- summed here, in
// slice order, rounded to bf16 (what that linear would have stored).
struct AttnSource {
  uint16_t *in;
  int ld, S;
  const float *part;
  size_t n, slice;
  uint16_t qw[2], kw[2];  // this lane's norm weights
};
// Rows [0, n) by the workgroup, RF per wavefront in flight.  Bound by round trips: everything a row needs is requested before the first
// value is waited for (the row, then its norm weights, then its rotation had made it three, and a branch around each row as many more).
// own(tok): an unsummed row of this token is also stored where the linear would have.
template <int RF, int NW = MK_WAVES, typename Row, typename Own>
__device__ __forceinline__ void attn_rows(CStage &st, const AttnSource &src, int n, int lane, int wave, Row row, Own own) {
  for (int i0 = NW - 1 - wave; i0 < n; i0 += RF * NW) {
    AttnRow a[RF];
    uint16_t cs[RF], sn[RF];
    float x[RF][2];
#pragma unroll
    for (int r = 0; r < RF; r++) a[r] = row(min(i0 + r * NW, n - 1));
    if (st.flags & MK_F_ROPE) {
#pragma unroll
      for (int r = 0; r < RF; r++) {
        cs[r] = ((const uint16_t *)st.cos_tab + (size_t)a[r].pos * st.ld_cos)[lane];
        sn[r] = ((const uint16_t *)st.sin_tab + (size_t)a[r].pos * st.ld_cos)[lane];
      }
    }
    auto sum = [&](auto ns) {
      constexpr int NS = decltype(ns)::value;
      float q[RF][2][NS];
#pragma unroll
      for (int r = 0; r < RF; r++) {
        const float *pp = src.part + (size_t)a[r].tok * src.n + a[r].off + lane;
#pragma unroll
        for (int b = 0; b < NS; b++) {
          q[r][0][b] = ldc_f32(pp + b * src.slice);
          q[r][1][b] = ldc_f32(pp + b * src.slice + 64);
        }
      }
#pragma unroll
      for (int r = 0; r < RF; r++)
#pragma unroll
        for (int e = 0; e < 2; e++) {
          float v = 0.f;
#pragma unroll
          for (int b = 0; b < NS; b++) v += q[r][e][b];
          x[r][e] = bfround(v);
        }
    };
    if (src.S == 0) {
      uint16_t q[RF][2];
#pragma unroll
      for (int r = 0; r < RF; r++) {
        const uint16_t *pp = src.in + (size_t)a[r].tok * src.ld + a[r].off + lane;
        q[r][0] = ldc_u16(pp);
        q[r][1] = ldc_u16(pp + 64);
      }
#pragma unroll
      for (int r = 0; r < RF; r++) {
        x[r][0] = bf2f(q[r][0]);
        x[r][1] = bf2f(q[r][1]);
      }
    } else if (src.S == 2) {
      sum(std::integral_constant<int, 2>{});
    } else if (src.S == 4) {
      sum(std::integral_constant<int, 4>{});
    } else {
      sum(std::integral_constant<int, 8>{});
    }
#pragma unroll
    for (int r = 0; r < RF; r++) {
      if (i0 + r * NW >= n) break;
      float x0 = x[r][0], x1 = x[r][1];
      if (src.S && own(a[r].tok)) {
        uint16_t *d = src.in + (size_t)a[r].tok * src.ld + a[r].off;
        d[lane] = (uint16_t)f2bf(x0);
        d[lane + 64] = (uint16_t)f2bf(x1);
      }
      if (a[r].kind < 2) {
        if (st.flags & MK_F_QK_NORM) {
          const float ss = wave_sum(x0 * x0 + x1 * x1);
          const float f = rsqrtf(ss * (1.f / 128.f) + st.eps);
          x0 = bfround((x0 * f) * bf2f(a[r].kind ? src.kw[0] : src.qw[0]));
          x1 = bfround((x1 * f) * bf2f(a[r].kind ? src.kw[1] : src.qw[1]));
        }
        if (st.flags & MK_F_ROPE) {
          const float c_ = bf2f(cs[r]), s_ = bf2f(sn[r]);
          const float y0 = x0 * c_ - x1 * s_;
          const float y1 = x0 * s_ + x1 * c_;
          x0 = y0;
          x1 = y1;
        }
      }
      a[r].dst[lane] = (uint16_t)f2bf(x0);
      a[r].dst[lane + 64] = (uint16_t)f2bf(x1);
    }
  }
}
// (before the barrier: the norm weights; after it: where the rows are)
__device__ __forceinline__ AttnSource attn_source(CStage &st, int lane) {
  AttnSource s;
  if (st.flags & MK_F_QK_NORM) {
#pragma unroll
    for (int e = 0; e < 2; e++) {
      s.qw[e] = ((const uint16_t *)st.q_norm_w)[lane + 64 * e];
      s.kw[e] = ((const uint16_t *)st.k_norm_w)[lane + 64 * e];
    }
  }
  return s;
}
__device__ __forceinline__ void attn_source_ready(CStage &st, Ctx &c, AttnSource &s) {
  s.in = (uint16_t *)st.in;
  s.ld = st.ld_in;
  s.S = c.defer_S;
  s.part = c.defer_part;
  s.n = (size_t)c.defer_n;
  s.slice = (size_t)c.defer_rows * s.n;
  c.defer_S = 0;
}

#ifndef MK_TUNE_NPRE
#define MK_TUNE_NPRE 4
#endif
struct AttnUnit {
  int t, h, cidx, C, start, end, p, p0, t0, new_lo, n_new, cend;
  const int *pages;
};

// GQA decode attention with the q/k-norm, RoPE and KV append fused in front.  Work unit =
// (token, kv head, KV chunk); chunks of one (token, kv head) are adjacent virtual workgroups so a
// kv head stays on one XCD.  Inside a workgroup, sixteen 16-lane groups each walk every 16th
// position of the chunk with their own online-softmax state (fp32 running max / sum, exp2 with
// log2e folded into the scale); each lane owns 8 of the 128 head dims.  Groups are merged through
// LDS, chunks through an HBM workspace by the last workgroup to arrive.
//
// The cached K/V rows of a chunk do not depend on the running iteration (positions below the request's first new
// token were appended by earlier iterations), so the first unit's rows are requested BEFORE the grid barrier of the
// previous stage is awaited, like the weight rows of a linear.  They are read with ordinary loads: every iteration
// starts with a cache invalidate, rows are line-aligned per (position, head), and a row is never read in the
// iteration that writes it (the new positions come from LDS).
// Reference tasks: kv_cache_update_impl (tasks/mi300/kv_cache_update_mi300.cuh:41-327),
// paged_attention_minimal_decode (tasks/mi300/paged_attention_decode_minimal_mi300.cuh:100-371),
// gang_attention_split_kv_kernel (tasks/mi300/gang_attention_mi300.cuh:49-153).
template <int QPK>
__device__ __forceinline__ void stage_attn(CStage &st, Ctx &c, const MkRuntime &rt, int M, char *smem) {
  constexpr int D = 128;
  constexpr int NPRE = MK_TUNE_NPRE;          // positions per lane group requested ahead
  constexpr int DPT = QPK * D / MK_THREADS;   // merged outputs per thread (all of one head)
  constexpr int TPH = D / DPT;                // threads per head in the merges
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j16 = lane & 15, gg = wave * 4 + (lane >> 4);
  const int nkv = st.num_kv_heads;
  // LDS: q rows, then the K and V rows of this iteration's new positions (a request ingests up to MK_MAX_NEW_PER_REQ prompt
  // tokens per iteration), then the per-group partial results
  uint16_t *qs = (uint16_t *)smem;                                        // [QPK][128]
  int *sflag = (int *)(smem + 2048);
  uint16_t *knew = (uint16_t *)(smem + 4096);                             // [MK_MAX_NEW_PER_REQ][128]
  uint16_t *vnew = knew + MK_MAX_NEW_PER_REQ * D;                         // [MK_MAX_NEW_PER_REQ][128]
  constexpr int NG = 16;
  constexpr int PART_OFF = 4096 + 2 * MK_MAX_NEW_PER_REQ * D * 2;
  float *part = (float *)(smem + PART_OFF);  // [NG][QPK][132]
  static_assert(PART_OFF + NG * QPK * 132 * 4 <= MK_LDS_BYTES, "attention scratch exceeds the LDS window");
  const int n_items = M * nkv;
  int cmax = c.G / n_items;
  cmax = cmax < 1 ? 1 : (cmax > MK_ATTN_MAX_CHUNKS ? MK_ATTN_MAX_CHUNKS : cmax);
  const int n_units = n_items * cmax;
  const int ps = rt.page_size;
  const u32x4 *kc = (const u32x4 *)st.k_cache;
  const u32x4 *vc = (const u32x4 *)st.v_cache;

  auto decode = [&](int u, AttnUnit &a) -> bool {
    const int item = u / cmax;
    a.cidx = u - item * cmax;
    a.t = item / nkv;
    a.h = item - a.t * nkv;
    a.p = __builtin_amdgcn_readfirstlane(c.sh_tok[a.t]);
    const int L = a.p + 1;
    a.t0 = __builtin_amdgcn_readfirstlane(c.sh_tok[2 * MK_MAX_TOKENS + a.t]);
    a.p0 = __builtin_amdgcn_readfirstlane(c.sh_tok[a.t0]);
    const int Lc = min(a.p0, L);  // cached positions this token sees
    // Up to 64 cached positions (4 per lane group: one block) per chunk.  While workgroups are plenty, one more chunk
    // takes this iteration's new positions and nothing else: that chunk also prepares their K/V rows and appends the
    // newest one, which would otherwise make it the last to finish.
    const int Cd = (Lc + 63) / 64 + 1;
    const bool own_chunk = L > 64 && Cd <= cmax;
    int C = own_chunk ? Cd : (L + 63) / 64;
    a.C = C > cmax ? cmax : C;
    if (a.cidx >= a.C) return false;
    if (own_chunk) {
      const int nc = a.C - 1;
      a.start = a.cidx < nc ? (int)(((long long)Lc * a.cidx) / nc) : Lc;
      a.end = a.cidx < nc ? (int)(((long long)Lc * (a.cidx + 1)) / nc) : L;
    } else {
      a.start = (int)(((long long)L * a.cidx) / a.C);
      a.end = (int)(((long long)L * (a.cidx + 1)) / a.C);
    }
    a.pages = rt.kv_indices + __builtin_amdgcn_readfirstlane(c.sh_tok[3 * MK_MAX_TOKENS + a.t]);
    a.new_lo = max(a.start, a.p0);  // new positions handled here: [new_lo, end)
    a.n_new = a.end > a.new_lo ? a.end - a.new_lo : 0;
    a.cend = min(a.end, a.p0);      // cached positions handled here: [start, cend)
    return true;
  };
  auto kvoff = [&](const AttnUnit &a, int pos) -> size_t {
    const int pg = pos / ps;
    const size_t row = (size_t)a.pages[pg] * ps + (pos - pg * ps);
    return (row * nkv + a.h) * (D / 8) + j16;
  };

  // ---- before the barrier: the first unit's cached rows
  AttnUnit a0;
  const bool have0 = c.vid < n_units && decode(c.vid, a0);
  u32x4 pk[NPRE], pv[NPRE];
  auto prefetch0 = [&]() {
#pragma unroll
    for (int i = 0; i < NPRE; i++) {
      const int pos = a0.start + gg + 16 * i;
      if (pos < a0.cend) {
        const size_t off = kvoff(a0, pos);
        pk[i] = kc[off];
        pv[i] = vc[off];
      }
    }
  };
  // the polling wavefront keeps its memory queue empty until the barrier is through (its loads would delay the poll
  // results behind them); its rows are requested right after and land while the q rows are being fetched
  if (have0 && wave != 0) prefetch0();
  AttnSource src = attn_source(st, lane);
  barrier_wait(c);
  if (have0 && wave == 0) prefetch0();
  attn_source_ready(st, c, src);

  for (int uu = c.vid; uu < n_units; uu += c.G) {
    AttnUnit a;
    const bool first = uu == c.vid;
    // More (token, kv head) pairs than workgroups: every other round deals them in reverse order, so a workgroup that
    // drew a long context in one round draws from the other end of the batch in the next (requests that entered the
    // batch together sit next to each other and are about equally far along).
    int u = uu;
    if (cmax == 1 && ((uu / c.G) & 1)) {
      const int r0 = (uu / c.G) * c.G, rn = min(c.G, n_units - r0);
      u = r0 + rn - 1 - (uu - r0);
    }
    if (first) {
      if (!have0) continue;
      a = a0;
    } else if (!decode(u, a)) {
      continue;
    }
    const int t = a.t, h = a.h, p = a.p, C = a.C;
    __syncthreads();  // LDS reuse across units
    // ---- phase A: prepare q heads and the new K/V rows of this chunk
    attn_rows<QPK == 8 ? 3 : 2>(st, src, QPK + 2 * a.n_new, lane, wave,  // (the rows of one new position in one round trip)
                 [&](int i) -> AttnRow {
                   const int j = i - QPK, kind = j < 0 ? 0 : j < a.n_new ? 1 : 2, jj = kind == 2 ? j - a.n_new : j, base = h * (QPK + 2) * D;
                   return kind ? AttnRow{a.t0 + (a.new_lo + jj - a.p0), base + (QPK + kind - 1) * D, a.new_lo + jj, kind, (kind == 1 ? knew : vnew) + jj * D}
                               : AttnRow{t, base + i * D, p, 0, qs + i * D};
                 },
                 [&](int tok) { return a.cidx == C - 1 && tok == t; });
    __syncthreads();
    // the chunk that owns the newest position appends this token's K/V and publishes q
    if (a.cidx == C - 1) {
      const int j = p - a.new_lo;
      const size_t rowi = (size_t)a.pages[p / ps] * ps + (p % ps);
      uint32_t *kd = (uint32_t *)st.k_cache + (rowi * nkv + h) * (D / 2);
      uint32_t *vd = (uint32_t *)st.v_cache + (rowi * nkv + h) * (D / 2);
      if (tid < 64) kd[tid] = ((const uint32_t *)(knew + j * D))[tid];
      else if (tid < 128) vd[tid - 64] = ((const uint32_t *)(vnew + j * D))[tid - 64];
      if (st.q_ws) {
        uint32_t *qd = (uint32_t *)st.q_ws + ((size_t)t * st.ld_qws + (size_t)h * QPK * D) / 2;
        for (int i = tid; i < QPK * D / 2; i += MK_THREADS) qd[i] = ((const uint32_t *)qs)[i];
      }
    }
    MK_MARK(c, first ? 0 : 2);
    // ---- phase B: online softmax over the chunk
    u32x4 qv[QPK];
#pragma unroll
    for (int hh = 0; hh < QPK; hh++) qv[hh] = ((const u32x4 *)qs)[hh * 16 + j16];
    float m[QPK], l[QPK], acc[QPK][8];
#pragma unroll
    for (int hh = 0; hh < QPK; hh++) {
      m[hh] = -INFINITY;
      l[hh] = 0.f;
#pragma unroll
      for (int d = 0; d < 8; d++) acc[hh][d] = 0.f;
    }
    auto process = [&](const u32x4 kv, const u32x4 vv) {
      float v[8] = {bf_lo(vv.x), bf_hi(vv.x), bf_lo(vv.y), bf_hi(vv.y), bf_lo(vv.z), bf_hi(vv.z), bf_lo(vv.w), bf_hi(vv.w)};
#pragma unroll
      for (int hh = 0; hh < QPK; hh++) {
        float s = group16_sum(dot8(kv, qv[hh], 0.f)) * st.sm_scale_log2;
        const float mn = fmaxf(m[hh], s);
        const float alpha = __builtin_amdgcn_exp2f(m[hh] - mn);
        const float pr = __builtin_amdgcn_exp2f(s - mn);
        l[hh] = l[hh] * alpha + pr;
#pragma unroll
        for (int d = 0; d < 8; d++) acc[hh][d] = acc[hh][d] * alpha + pr * v[d];
        m[hh] = mn;
      }
    };
    // NPRE positions at a time: all scores first (independent reductions), then ONE rescale of the running state.
    // Entries at or beyond cend hold whatever the registers held; their scores are forced to -inf (weight 0).
    auto process_block = [&](const u32x4 (&kk)[NPRE], const u32x4 (&vv)[NPRE], int pos0) {
      float sc[NPRE][QPK];  // scores, then softmax weights
#pragma unroll
      for (int i = 0; i < NPRE; i++) {
        const bool ok = pos0 + 16 * i < a.cend;
#pragma unroll
        for (int hh = 0; hh < QPK; hh++) {
          const float d = group16_sum(dot8(kk[i], qv[hh], 0.f)) * st.sm_scale_log2;
          sc[i][hh] = ok ? d : -INFINITY;
        }
      }
#pragma unroll
      for (int hh = 0; hh < QPK; hh++) {
        float mn = m[hh];
#pragma unroll
        for (int i = 0; i < NPRE; i++) mn = fmaxf(mn, sc[i][hh]);
        const float alpha = __builtin_amdgcn_exp2f(m[hh] - mn);
        float ps_ = 0.f;
#pragma unroll
        for (int i = 0; i < NPRE; i++) {
          sc[i][hh] = __builtin_amdgcn_exp2f(sc[i][hh] - mn);
          ps_ += sc[i][hh];
        }
        l[hh] = l[hh] * alpha + ps_;
        m[hh] = mn;
#pragma unroll
        for (int d = 0; d < 8; d++) acc[hh][d] *= alpha;
      }
#pragma unroll
      for (int i = 0; i < NPRE; i++) {
        const bool ok = pos0 + 16 * i < a.cend;
        const u32x4 w = vv[i];
        float v[8] = {bf_lo(w.x), bf_hi(w.x), bf_lo(w.y), bf_hi(w.y), bf_lo(w.z), bf_hi(w.z), bf_lo(w.w), bf_hi(w.w)};
#pragma unroll
        for (int d = 0; d < 8; d++) v[d] = ok ? v[d] : 0.f;  // 0 * NaN from an unloaded register would poison the sum
#pragma unroll
        for (int hh = 0; hh < QPK; hh++) {
#pragma unroll
          for (int d = 0; d < 8; d++) acc[hh][d] += sc[i][hh] * v[d];
        }
      }
    };
    int pos = a.start + gg;
    if (first) {
      if (pos < a.cend) process_block(pk, pv, pos);
      pos += 16 * NPRE;
    }
    // later blocks: the next block's rows are in flight while the current one is reduced
    // Every load is issued unconditionally (positions beyond the chunk re-read its last row and are masked in
    // process_block): a load under a branch would turn the wait for the current block into a wait for the next one too.
    auto load_block = [&](int p0, u32x4 (&kk)[NPRE], u32x4 (&vv)[NPRE]) {
#pragma unroll
      for (int i = 0; i < NPRE; i++) {
        const size_t off = kvoff(a, min(p0 + 16 * i, a.cend - 1));
        kk[i] = kc[off];
        vv[i] = vc[off];
      }
    };
    if (pos < a.cend) {
      u32x4 ka[NPRE], va[NPRE], kb[NPRE], vb[NPRE];
      load_block(pos, ka, va);
      while (true) {
        load_block(pos + 16 * NPRE, kb, vb);
        process_block(ka, va, pos);
        pos += 16 * NPRE;
        if (pos >= a.cend) break;
        load_block(pos + 16 * NPRE, ka, va);
        process_block(kb, vb, pos);
        pos += 16 * NPRE;
        if (pos >= a.cend) break;
      }
    }
    for (int j = gg; j < a.n_new; j += 16) process(((const u32x4 *)(knew + j * D))[j16], ((const u32x4 *)(vnew + j * D))[j16]);
    // ---- phase C: merge the 16 groups through LDS
#pragma unroll
    for (int hh = 0; hh < QPK; hh++) {
      float *pp = part + (gg * QPK + hh) * 132;
#pragma unroll
      for (int d = 0; d < 8; d++) pp[j16 * 8 + d] = acc[hh][d];
      if (j16 == 0) {
        pp[128] = m[hh];
        pp[129] = l[hh];
      }
    }
    __syncthreads();
    // When every chunk of this (token, kv head) runs on one die, the partials and the arrival counter never leave that
    // die's L2: workgroup-scope atomic, ordinary stores and loads (each stage has its own partial buffer and the L1 is
    // invalidated once per iteration, so a partial is never read from a stale line).  Otherwise device scope.
    const int item = u / cmax;
    // (a launch whose attention stages all share one partial buffer -- rt.attn_part -- always takes the device-scope
    // path: a buffer that is rewritten several times per iteration must not be read through lines an earlier stage left
    // in the L1)
    const bool local = !rt.attn_part && c.even_xcds && (item * cmax) / c.quota == (item * cmax + C - 1) / c.quota;
    float *part_base = rt.attn_part ? rt.attn_part : (float *)st.aux0;
    float *gpart = part_base + (size_t)u * QPK * MK_ATTN_PSTRIDE;
    uint16_t *orow = (uint16_t *)st.out + (size_t)t * st.ld_out + (size_t)h * QPK * D;
    const int mh = tid / TPH, md = (tid - mh * TPH) * DPT;  // this thread merges dims [md, md+DPT) of head mh
    {
      float mx = -INFINITY;
#pragma unroll
      for (int g = 0; g < NG; g++) mx = fmaxf(mx, part[(g * QPK + mh) * 132 + 128]);
      float ls = 0.f, os[DPT];
#pragma unroll
      for (int d = 0; d < DPT; d++) os[d] = 0.f;
#pragma unroll
      for (int g = 0; g < NG; g++) {
        const float *pp = part + (g * QPK + mh) * 132;
        const float wgt = __builtin_amdgcn_exp2f(pp[128] - mx);
        ls += pp[129] * wgt;
#pragma unroll
        for (int d = 0; d < DPT; d++) os[d] += pp[md + d] * wgt;
      }
      if (C == 1) {
#pragma unroll
        for (int d = 0; d < DPT; d += 2)  // written through: the stage's barrier skips the L2 write-back
          __hip_atomic_store((uint32_t *)(orow + mh * D + md + d), pack2(os[d] / ls, os[d + 1] / ls), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        // 8-byte stores that together cover whole 128-byte lines (the running max and sum fill a line of their own, 16
        // copies), so that the merging workgroup never reads a line that is only partly valid in the L2
#pragma unroll
        for (int d = 0; d < DPT; d += 2) *(float2 *)(gpart + mh * MK_ATTN_PSTRIDE + md + d) = make_float2(os[d], os[d + 1]);
        if (md < 16 * DPT) *(float2 *)(gpart + mh * MK_ATTN_PSTRIDE + D + 2 * (md / DPT)) = make_float2(mx, ls);
      }
    }
    if (C > 1) {
      // ---- phase D: the last chunk to finish merges all chunks of this (token, kv head)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) {
        int last;
        if (local) {
          unsigned *cnt = (unsigned *)st.aux1 + (size_t)item * 32;
          last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP) == (unsigned)(C - 1);
          if (last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        } else {
          unsigned *cnt = &rt.attn_cnt[(size_t)item * 32];
          last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(C - 1);
          if (last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        *sflag = last;
      }
      __syncthreads();
      if (*sflag) {
        // every chunk partial is read with independent loads (8 bytes each), sixteen chunks in flight per thread
        const float *ip = part_base + (size_t)item * cmax * QPK * MK_ATTN_PSTRIDE;
        float mx = -INFINITY, ls = 0.f, os[DPT];
#pragma unroll
        for (int d = 0; d < DPT; d++) os[d] = 0.f;
        auto merge16 = [&](int c0, auto load8) {
          float2 ml[16], ov[16][DPT / 2];
#pragma unroll
          for (int j = 0; j < 16; j++) {
            if (c0 + j < C) {
              const float *pp = ip + ((size_t)(c0 + j) * QPK + mh) * MK_ATTN_PSTRIDE;
              ml[j] = load8(pp + D);
#pragma unroll
              for (int d = 0; d < DPT / 2; d++) ov[j][d] = load8(pp + md + 2 * d);
            }
          }
#pragma unroll
          for (int j = 0; j < 16; j++)
            if (c0 + j < C) {
              const float mn = fmaxf(mx, ml[j].x);
              const float sa = __builtin_amdgcn_exp2f(mx - mn), sb = __builtin_amdgcn_exp2f(ml[j].x - mn);
              ls = ls * sa + ml[j].y * sb;
#pragma unroll
              for (int d = 0; d < DPT / 2; d++) {
                os[2 * d] = os[2 * d] * sa + ov[j][d].x * sb;
                os[2 * d + 1] = os[2 * d + 1] * sa + ov[j][d].y * sb;
              }
              mx = mn;
            }
        };
        if (local) {
          for (int c0 = 0; c0 < C; c0 += 16) merge16(c0, [](const float *q) { return *(const float2 *)q; });
        } else {
          for (int c0 = 0; c0 < C; c0 += 16)
            merge16(c0, [](const float *q) {
              const unsigned long long u = ldc_u64(q);
              return make_float2(__uint_as_float((uint32_t)u), __uint_as_float((uint32_t)(u >> 32)));
            });
        }
#pragma unroll
        for (int d = 0; d < DPT; d += 2)  // written through: the stage's barrier skips the L2 write-back
          __hip_atomic_store((uint32_t *)(orow + mh * D + md + d), pack2(os[d] / ls, os[d + 1] / ls), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  // The attention outputs went through to memory.  The appended K/V rows and the published q rows stay in this die's
  // L2 until something writes it back: the barrier behind the scheduler step that opens the next iteration, or the end of the launch.  (No
  // later stage of this iteration needs to.)  Nothing reads them before the next iteration.
  c.wrote_through = true;
}


#define MK_ATTN_PAIR_PAGES 1024  // page-table entries of a request where a workgroup works on two units at a time
// Whether a workgroup takes two units at a time (below).  One after the other, its units take as many turns as the workgroup has; two at a time
// half of them, rounded up, which last as long as the longer of the two and walk a context with two wavefronts instead of four.  So pairs save
// what a turn costs besides its positions (420 positions' worth, 320 with eight queries a head, of which two wavefronts prepare twice as many)
// and lose 0.95 of every position that the second unit does not have as well, and half a turn where the number of turns is odd.  The longest turn of
// pairs is taken to be the longest context's, the others average ones; a workgroup that takes one after the other is taken to walk average
// contexts, or the longest one, whichever is more.  (With the shortest contexts beside the longest, or with the sum in one place for both query
// counts, the rule is no better and the linears of the same kernel get other registers: 3 to 25 tokens of qwen3-8b 0.6 to 0.9 % slower.)
// As a stage of 64 requests, us, one after the other -> two at a time.  Two turns (8 kv heads, 4 queries): contexts of 320 29.5 -> 21.8, 1000 54.5 ->
// 48.4, 1480 73.5 -> 66.8; of 1000 .. 1480 66.2 -> 63.9, 100 .. 700 34.4 -> 34.4, 100 .. 850 36.6 -> 40.1, 1000 .. 1700 69.3 -> 70.9; 63 of 20 and one
// of 390 25.3 -> 23.7, of 900 33.6 -> 40.3.  Three turns (12 kv heads): 320 43.9 -> 39.1, 510 53.4 -> 53.3, 700 65.5 -> 67.3, 1000 83.5 -> 90.5, 100 .. 700
// 50.3 -> 53.1; with 8 queries 320 45.8 -> 44.8, 450 55.2 -> 56.8.  Four (16): 320 56.4 -> 40.9, 1480 149.5 -> 136.4, 100 .. 850 70.4 -> 65.5, 100 .. 1480
// 94.3 -> 95.3.  Five (20): 700 108.6 -> 102.4, 1000 136.9 -> 137.9, 1480 185.7 -> 190.0.  (By the longest context's distance from the average, 384,
// three turns of 1000 and 1480 positions had become 10 % and 12 % slower than one unit after the other, two turns of 100 .. 850 9 %.)
template <int QPK>
__device__ __forceinline__ bool attn_in_pairs(CStage &st, const Ctx &c, const MkRuntime &rt, int M) {
  const int lane = threadIdx.x & 63, first = lane < M ? c.sh_tok[2 * MK_MAX_TOKENS + lane] : 0;
  const int units = __popcll(__ballot(lane < M && (lane - first) % (16 / QPK) == 0)) * st.num_kv_heads, turns = (units + c.G - 1) / c.G, pairs = (turns + 1) / 2;
  if (turns < 2 || (rt.max_seq + rt.page_size - 1) / rt.page_size > MK_ATTN_PAIR_PAGES) return false;
  const int pos = lane < M ? c.sh_tok[lane] : 0;
  const float mean = wave_sum((float)pos) / (float)M;
  const float save = (QPK == 4 ? 420.f : 320.f) * (float)(turns - pairs) - 1.95f * (float)(pairs - 1) * mean;
  return !__any((float)pos > fmaxf((save + (float)turns * mean) * (1.f / 1.95f), save * (1.f / 0.95f)));
}

// The same for iterations of many tokens, on the matrix cores.  Work unit = (up to 16 / QPK consecutive tokens of one request, kv head,
// KV chunk): their query rows are the 16 columns of a tile product, so a prompt's tokens share what is read of the cache.  One wavefront
// per tile of 16 positions; the new positions of the iteration are tiles as well, out of LDS.
//
// Bound by the cache's way through L2 for long prompts and by round trips for short contexts.  A unit per token had read the cache once
// for every token of a prompt and prepared its new key rows as often.  64 tokens of one prompt, 32 q / 8 kv heads, as a stage: behind 1216
// cached positions 85 -> 31 us, behind 2432 127 -> 43; 64 streams of one token 33 -> 32.  (A portion at the very start of its prompt is as fast as
// before or, with few kv heads, slower, its new rows being prepared by fewer workgroups: 64 tokens of 8 q / 2 kv heads 29 -> 32.)
//
// Tile: scores with A = K (lane (i, g): row of position i, dims 32 s + 8 g .. of step s) and B = q (lane (j, g): column j, same dims)
// -> lane (j, g) holds column j at positions 4 g .. 4 g + 3.  Those four weights are already the A operand of a 16x16x16 step over
// positions, in bf16 terms: cached positions as value and rounding remainder (two operands, 16 bits of a weight), new ones, of which there
// are few tiles, with all of their 24 bits (three).  The B operand -- four consecutive positions of one dim -- is read out of the V tile in LDS.  The running maximum is kept per column for the whole wavefront, the running sum per lane.
// K and V tiles are four groups of four rows of 256 bytes, one direct-to-LDS request per group (each lane 16 bytes: four whole rows), the
// groups GS bytes apart (the transposed V reads of the four groups then fall into different banks).
template <int QPK, bool PAIR>
__device__ __forceinline__ void stage_attn_tiles(CStage &st, Ctx &c, const MkRuntime &rt, int M, char *smem) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  constexpr int D = 128, NC = 16, TG = NC / QPK, RB = 2, PD = 132;
  constexpr int SUBS = PAIR ? 2 : 1, SW = MK_WAVES / SUBS, ST = SW * 64;  // units at a time, wavefronts and threads of one
  constexpr int GS = 1088, TS = 4 * GS, SLOT = 2 * TS, NEW_BYTES = MK_MAX_NEW_PER_REQ / 4 * GS;
  // LDS: query rows, new rows and page list of every unit, then the tiles of every wavefront.  The wavefronts' partial results have an area
  // of their own, which the page list shares, or, with two units, lie where the wavefront's tiles were.
  constexpr int FLAG_OFF = SUBS * NC * D * 2, KN_OFF = FLAG_OFF + 64, PART_OFF = KN_OFF + SUBS * 2 * NEW_BYTES;
  constexpr int BUF_OFF = PART_OFF + (PAIR ? SUBS * MK_ATTN_PAIR_PAGES * 4 : MK_WAVES * NC * PD * 4);
  static_assert(BUF_OFF + MK_WAVES * RB * SLOT <= MK_LDS_BYTES, "attention scratch exceeds the LDS window");
  static_assert(MK_ATTN_MAX_REQ_PAGES * 4 <= MK_WAVES * NC * PD * 4, "page list exceeds the area it aliases");
  static_assert(NC * PD * 4 <= RB * SLOT, "partial results exceed the tiles they follow");
  static_assert(PART_OFF % 16 == 0 && BUF_OFF % 16 == 0 && KN_OFF % 16 == 0, "16-byte operands");
  const int tid = c.tid, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;
  const int sub = wave / SW, sw = wave % SW, stid = tid % ST;  // which unit, wavefront and thread of it
  const int nkv = st.num_kv_heads, ps = rt.page_size;
  uint16_t *qs = (uint16_t *)smem + sub * NC * D;                  // [16][128]
  int *sflag = (int *)(smem + FLAG_OFF);
  char *knew = smem + KN_OFF + sub * 2 * NEW_BYTES, *vnew = knew + NEW_BYTES;  // new rows as tiles
  auto part_of = [&](int w) { return (float *)(smem + (PAIR ? BUF_OFF + (sub * SW + w) * (RB * SLOT) : PART_OFF + w * NC * PD * 4)); };  // [16][PD]: values, maximum, sum
  int *spg = (int *)(smem + PART_OFF) + (PAIR ? sub * MK_ATTN_PAIR_PAGES : 0);  // page list of the running unit (until the partials are written)
  char *buf = smem + BUF_OFF + wave * (RB * SLOT);
  const u32x4 *kc = (const u32x4 *)st.k_cache, *vc = (const u32x4 *)st.v_cache;
  auto new_row = [&](char *base, int j) { return (uint16_t *)(base + (j >> 2) * GS + (j & 3) * 256); };
  // groups of tokens: every TG-th token of a request begins one
  const int my_first = lane < M ? c.sh_tok[2 * MK_MAX_TOKENS + lane] : 0;
  const unsigned long long begins = __ballot(lane < M && (lane - my_first) % TG == 0);
  const int groups = __popcll(begins), n_items = groups * nkv;
  const int cmax = max(1, min(c.G / n_items, MK_ATTN_MAX_CHUNKS)), n_units = n_items * cmax;
  struct Unit {
    int item, cidx, C, t, n, h, p0, p, t0, tb, te, n_new;
    const int *pages;
  };
  auto decode = [&](int u, Unit &a) -> bool {
    a.item = u / cmax;
    a.cidx = u - a.item * cmax;
    const int g = a.item / nkv;
    a.h = a.item - g * nkv;
    const bool mine = ((begins >> lane) & 1) && __popcll(begins & ((1ull << lane) - 1)) == g;
    a.t = (int)__ffsll(__ballot(mine)) - 1;
    a.t0 = __builtin_amdgcn_readfirstlane(c.sh_tok[2 * MK_MAX_TOKENS + a.t]);
    a.n = __popcll(__ballot(lane < M && lane >= a.t && lane < a.t + TG && my_first == a.t0));
    a.p0 = __builtin_amdgcn_readfirstlane(c.sh_tok[a.t0]);
    a.p = __builtin_amdgcn_readfirstlane(c.sh_tok[a.t]) + a.n - 1;  // newest position
    const int nt = (a.p0 + 15) / 16, n_new = a.p + 1 - a.p0;        // cached tiles, new rows
    // One cached tile per wavefront and a chunk of its own for the new rows while workgroups are plenty; else the last chunk, which
    // prepares those rows, takes fewer tiles: a round of rows takes as long as about four tiles of every wavefront.
    const int Cd = (nt + MK_WAVES - 1) / MK_WAVES + 1;
    a.C = min(Cd, cmax);
    if (a.cidx >= a.C) return false;
    if (a.C == Cd) {
      a.tb = a.cidx < a.C - 1 ? (int)((long long)nt * a.cidx / (a.C - 1)) : nt;
      a.te = a.cidx < a.C - 1 ? (int)((long long)nt * (a.cidx + 1) / (a.C - 1)) : nt;
    } else {
      const int extra = 4 * MK_WAVES * ((a.n * QPK + 2 * n_new + 31) / 32 - 1);
      const int total = nt + (a.C > 1 ? min(extra, (nt + a.C - 2) / (a.C - 1)) : 0);
      a.tb = min(nt, (int)((long long)total * a.cidx / a.C));
      a.te = a.cidx < a.C - 1 ? min(nt, (int)((long long)total * (a.cidx + 1) / a.C)) : nt;
    }
    a.n_new = a.cidx == a.C - 1 ? n_new : 0;
    a.pages = rt.kv_indices + __builtin_amdgcn_readfirstlane(c.sh_tok[3 * MK_MAX_TOKENS + a.t]);
    return true;
  };
  // The page list of a workgroup's next unit is requested while it works on the one before, the first one's -- like the norm weights --
  // before the barrier is awaited.
  AttnSource src = attn_source(st, lane);
  auto page_range = [&](const Unit &a, int &lo) -> int {
    lo = a.tb * 16 / ps;
    return a.te > a.tb ? (min(a.p0, a.te * 16) - 1) / ps - lo + 1 : 0;
  };
  Unit next;
  int u_next, pg_next = 0;
  bool have = false;
  auto announce = [&](int uu) {
    u_next = uu;
    if (cmax == 1 && ((uu / c.G) & 1)) {  // every other round deals the units in reverse order (contexts differ)
      const int r0 = (uu / c.G) * c.G, rn = min(c.G, n_units - r0);
      u_next = r0 + rn - 1 - (uu - r0);
    }
    have = uu < n_units && decode(u_next, next);
    int lo;
    if (have && stid < page_range(next, lo)) pg_next = next.pages[lo + stid];
  };
  announce(c.vid + sub * c.G);
  barrier_wait(c);
  attn_source_ready(st, c, src);

  for (int uu = c.vid + sub * c.G; uu - sub * c.G < n_units; uu += SUBS * c.G) {
    if (!PAIR && !have) {
      announce(uu + c.G);
      continue;
    }
    Unit a = next;
    if (PAIR && !have) a.n = a.n_new = a.tb = a.te = 0;  // (the pair's other half has a unit: this one keeps the barriers)
    const int u = u_next;
    const int n_cols = a.n * QPK, p_first = a.p + 1 - a.n, nt = a.te - a.tb, cend = min(a.p0, a.te * 16);
    __syncthreads();  // LDS reuse across units
    // ---- page list, then the first tiles, then the rows
    int pg_lo;
    const int npg = page_range(a, pg_lo);
    if (stid < npg) spg[stid] = pg_next;
    for (int i = stid + ST; i < npg; i += ST) spg[i] = a.pages[pg_lo + i];
    for (int j = a.n_new * 16 + stid; j < (a.n_new + 15) / 16 * 256; j += ST) ((u32x4 *)new_row(vnew, j >> 4))[j & 15] = (u32x4){0u, 0u, 0u, 0u};
    __syncthreads();
    auto row_base = [&](int pos) -> size_t {  // first 16-byte operand of the (position, head) row
      const int pc = min(pos, cend - 1), pg = pc / ps;
      return (((size_t)spg[pg - pg_lo] * ps + (pc - pg * ps)) * nkv + a.h) * (D / 8);
    };
    // request s brings rows 4 s .. 4 s + 3 whole (lane (row in group, 16-byte piece)); streaming requests: a cached row need not displace
    // the activations the linears share through the L2.  A tile index past the end re-reads the last tile; it is never computed.
    auto load_tile = [&](int tt, char *b) {
      constexpr int KV_NT = 2;
      const int q0 = (a.tb + min(tt, nt - 1)) * 16;
      size_t gb[4];
#pragma unroll
      for (int s_ = 0; s_ < 4; s_++) gb[s_] = row_base(q0 + 4 * s_ + lg) + lr;
#pragma unroll
      for (int s_ = 0; s_ < 4; s_++)
        __builtin_amdgcn_global_load_lds((const MK_GLOBAL void *)(unsigned long long)(kc + gb[s_]),
                                         (__attribute__((address_space(3))) void *)(__attribute__((address_space(3))) char *)(b + TS + s_ * GS), 16, 0, KV_NT);
#pragma unroll
      for (int s_ = 0; s_ < 4; s_++)
        __builtin_amdgcn_global_load_lds((const MK_GLOBAL void *)(unsigned long long)(vc + gb[s_]),
                                         (__attribute__((address_space(3))) void *)(__attribute__((address_space(3))) char *)(b + s_ * GS), 16, 0, KV_NT);
    };
    if (sw < nt) {
#pragma unroll
      for (int b_ = 0; b_ < RB - 1; b_++) load_tile(sw + b_ * SW, buf + b_ * SLOT);
    }
    announce(uu + SUBS * c.G);
    auto row = [&](int i) -> AttnRow {
      const int j = i - n_cols, kind = j < 0 ? 0 : j < a.n_new ? 1 : 2, jj = kind == 2 ? j - a.n_new : j, base = a.h * (QPK + 2) * D;
      return kind ? AttnRow{a.t0 + jj, base + (QPK + kind - 1) * D, a.p0 + jj, kind, new_row(kind == 1 ? knew : vnew, jj)}
                  : AttnRow{a.t + i / QPK, base + (i % QPK) * D, p_first + i / QPK, 0, qs + i * D};
    };
    auto own = [&](int tok) { return a.n_new > 0 && tok >= a.t; };
    const int n_rows = n_cols + 2 * a.n_new;
    if (n_rows > 4 * SW) attn_rows<8, SW>(st, src, n_rows, lane, sw, row, own);
    else attn_rows<4, SW>(st, src, n_rows, lane, sw, row, own);
    __syncthreads();
    // ---- tiles
    bf16x8 qb[4];
#pragma unroll
    for (int s_ = 0; s_ < 4; s_++) {
      const u32x4 z = {0u, 0u, 0u, 0u};
      qb[s_] = __builtin_bit_cast(bf16x8, lr < n_cols ? *(const u32x4 *)(qs + lr * D + s_ * 32 + lg * 8) : z);
    }
    f32x4 o[8];
#pragma unroll
    for (int dt = 0; dt < 8; dt++) o[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float mrun = -INFINITY, lsum = 0.f;
    // positions [q0, q0 + 16) whose rows lie at kb / vb; this lane's column sees those up to `last` (at least one of them)
    auto compute_tile = [&](int q0, int last, const char *kb, const char *vb, auto fresh) {
      constexpr bool NEW = decltype(fresh)::value;
      f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
      const char *kl = kb + (lr >> 2) * GS + (lr & 3) * 256 + lg * 16;
#pragma unroll
      for (int s_ = 0; s_ < 4; s_++) s4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, *(const u32x4 *)(kl + s_ * 64)), qb[s_], s4, 0, 0, 0);
      float sc[4];
#pragma unroll
      for (int r = 0; r < 4; r++) sc[r] = q0 + lg * 4 + r <= last ? s4[r] * st.sm_scale_log2 : -INFINITY;
      float mx = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
      mx = fmaxf(mx, __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 16) << 2, __builtin_bit_cast(int, mx))));
      mx = fmaxf(mx, __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __builtin_bit_cast(int, mx))));
      const float mn = fmaxf(mrun, mx);
      const float alpha = __builtin_amdgcn_exp2f(mrun - mn);
      float pw[4];
#pragma unroll
      for (int r = 0; r < 4; r++) pw[r] = __builtin_amdgcn_exp2f(sc[r] - mn);
      lsum = lsum * alpha + ((pw[0] + pw[1]) + (pw[2] + pw[3]));
      mrun = mn;
      if (__ballot(lr < n_cols && alpha != 1.f)) {  // (uniform) some column's maximum moved: rescale what has been summed
        float ar[4];
#pragma unroll
        for (int r = 0; r < 4; r++) ar[r] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lg * 4 + r) << 2, __builtin_bit_cast(int, alpha)));
#pragma unroll
        for (int dt = 0; dt < 8; dt++)
#pragma unroll
          for (int r = 0; r < 4; r++) o[dt][r] *= ar[r];
      }
      const char *vl = vb + lg * GS + lr * 2;
      if constexpr (NEW) {
        // A tile with a value that is not finite is summed column by column, each weight in one piece: zero times infinity is no number,
        // and zero is the weight of positions that only other columns see, and what is left behind the first term of many a weight.
        unsigned top = 0;
#pragma unroll
        for (int dt = 0; dt < 8; dt++) {
#pragma unroll
          for (int e = 0; e < 4; e++) top |= (*(const uint16_t *)(vl + dt * 32 + e * 256) & 0x7f80u) + 0x80u;
        }
        if (__builtin_expect(__ballot(top & 0x8000u) != 0, 0)) {
          for (int g = 0; g < 4; g++) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const uint16_t *v = (const uint16_t *)(vb + g * GS + e * 256) + lr;
#pragma unroll
              for (int r = 0; r < 4; r++) {
                const int col = lg * 4 + r;
                const float w = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((g * 16 + col) << 2, __builtin_bit_cast(int, pw[e])));
                const bool seen = q0 + g * 4 + e <= p_first + min(col, n_cols - 1) / QPK;
#pragma unroll
                for (int dt = 0; dt < 8; dt++) o[dt][r] = seen ? fmaf(w, bf2f(v[dt * 16]), o[dt][r]) : o[dt][r];
              }
            }
          }
          return;
        }
      }
      constexpr int NP = NEW ? 3 : 2;
      s16x4 wt[NP];
#pragma unroll
      for (int q = 0; q < NP; q++) {
        float ph[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          ph[r] = bfround(pw[r]);
          pw[r] -= ph[r];  // (exact)
        }
        wt[q] = __builtin_bit_cast(s16x4, (unsigned long long)pack2(ph[0], ph[1]) | ((unsigned long long)pack2(ph[2], ph[3]) << 32));
      }
#pragma unroll
      for (int dt = 0; dt < 8; dt++) {
        const char *q_ = vl + dt * 32;
        const unsigned v0 = *(const uint16_t *)(q_), v1 = *(const uint16_t *)(q_ + 256), v2 = *(const uint16_t *)(q_ + 512), v3 = *(const uint16_t *)(q_ + 768);
        const s16x4 bv = __builtin_bit_cast(s16x4, (unsigned long long)(v0 | (v1 << 16)) | ((unsigned long long)(v2 | (v3 << 16)) << 32));
#pragma unroll
        for (int q = 0; q < NP; q++) o[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wt[q], bv, o[dt], 0, 0, 0);
      }
    };
    // cached tiles: RB in flight per wavefront; every request is issued unconditionally, and the wait before a tile counts the
    // 8 (RB - 1) requests of the tiles after it
    int t_ = sw;
    if (t_ < nt) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (rows stored above are not counted below; the first tiles arrived with the rows)
      bool more = true;
      while (more) {
#pragma unroll
        for (int b_ = 0; b_ < RB; b_++) {
          load_tile(t_ + (RB - 1) * SW, buf + ((b_ + RB - 1) % RB) * SLOT);
          static_assert(RB == 2, "the wait counts one tile's requests");
          asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
          if (more) {
            compute_tile((a.tb + t_) * 16, cend - 1, buf + b_ * SLOT + TS, buf + b_ * SLOT, std::false_type{});
            t_ += SW;
            more = t_ < nt;
          }
        }
      }
    }
    // new tiles: all tokens of a group lie in the last of them (groups begin at multiples of TG in their request, TG divides 16)
    const int p_col = p_first + min(lr, n_cols - 1) / QPK;
    for (int k = sw; k * 16 < a.n_new; k += SW) compute_tile(a.p0 + k * 16, p_col, knew + k * TS, vnew + k * TS, std::true_type{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the direct-to-LDS requests of the tile that was not computed)
    // the chunk with the new rows appends the group's own K/V rows and publishes its queries
    if (a.n_new) {
      for (int i = stid; i < a.n * 64; i += ST) {
        const int pos = p_first + (i >> 6), e = i & 63;
        const size_t at = (((size_t)a.pages[pos / ps] * ps + pos % ps) * nkv + a.h) * (D / 2) + e;
        ((uint32_t *)st.k_cache)[at] = ((const uint32_t *)new_row(knew, pos - a.p0))[e];
        ((uint32_t *)st.v_cache)[at] = ((const uint32_t *)new_row(vnew, pos - a.p0))[e];
      }
      if (st.q_ws)
        for (int i = stid; i < n_cols * 64; i += ST) {
          const int col = i >> 6;
          ((uint32_t *)st.q_ws)[((size_t)(a.t + col / QPK) * st.ld_qws + (size_t)(a.h * QPK + col % QPK) * D) / 2 + (i & 63)] = ((const uint32_t *)qs)[i];
        }
    }
    if (!PAIR) __syncthreads();  // every wavefront is done with the page list: the partial results may overwrite it
    // ---- wavefronts
    float lt = lsum;
    lt += __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 16) << 2, __builtin_bit_cast(int, lt)));
    lt += __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __builtin_bit_cast(int, lt)));
    float *part = part_of(sw);
    if (lg == 0) {
      part[lr * PD + D] = mrun;
      part[lr * PD + D + 1] = lt;
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int dt = 0; dt < 8; dt++) part[(lg * 4 + r) * PD + dt * 16 + lr] = o[dt][r];
    __syncthreads();
    // (die-local or device-scope hand-over of chunks: see stage_attn)
    const bool local = !rt.attn_part && c.even_xcds && (a.item * cmax) / c.quota == (a.item * cmax + a.C - 1) / c.quota;
    float *part_base = rt.attn_part ? rt.attn_part : (float *)st.aux0;
    const int md = (tid & 15) * 8;  // this thread's dims; its column: one of sixteen, or, with two units at a time, two of theirs
    int col = stid >> 4;
    auto emit = [&](const float (&v)[8], float l) {  // written through: the stage's barrier skips the L2 write-back
      uint16_t *orow = (uint16_t *)st.out + (size_t)(a.t + col / QPK) * st.ld_out + (size_t)(a.h * QPK + col % QPK) * D + md;
#pragma unroll
      for (int d = 0; d < 8; d += 2) __hip_atomic_store((uint32_t *)(orow + d), pack2(v[d] / l, v[d + 1] / l), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto wavefronts = [&](float &mx, float &ls, float (&os)[8]) {  // the sum over the unit's wavefronts
      mx = -1e30f;
      ls = 0.f;
#pragma unroll
      for (int d = 0; d < 8; d++) os[d] = 0.f;
#pragma unroll
      for (int w = 0; w < SW; w++) mx = fmaxf(mx, part_of(w)[col * PD + D]);
#pragma unroll
      for (int w = 0; w < SW; w++) {
        const float *pp = part_of(w) + col * PD;
        const float wgt = __builtin_amdgcn_exp2f(pp[D] - mx);
        ls += pp[D + 1] * wgt;
#pragma unroll
        for (int d = 0; d < 8; d++) os[d] += pp[md + d] * wgt;
      }
    };
    if constexpr (PAIR) {
      for (; col < n_cols; col += ST / 16) {
        float mx, ls, os[8];
        wavefronts(mx, ls, os);
        emit(os, ls);
      }
      continue;
    }
    if (col < n_cols) {
      float mx, ls, os[8];
      wavefronts(mx, ls, os);
      if (a.C == 1) {
        emit(os, ls);
      } else {
        // whole 128-byte lines (the maximum and sum fill a line of their own, 16 copies): see stage_attn
        float *gp = part_base + ((size_t)u * NC + col) * MK_ATTN_PSTRIDE;
#pragma unroll
        for (int d = 0; d < 8; d += 4) *(f32x4 *)(gp + md + d) = (f32x4){os[d], os[d + 1], os[d + 2], os[d + 3]};
        *(float2 *)(gp + D + 2 * (tid & 15)) = make_float2(mx, ls);
      }
    }
    if (a.C == 1) continue;
    // ---- chunks: the last to finish merges them
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      int last;
      if (local) {
        unsigned *cnt = (unsigned *)st.aux1 + (size_t)a.item * 32;
        last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP) == (unsigned)(a.C - 1);
        if (last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      } else {
        unsigned *cnt = &rt.attn_cnt[(size_t)a.item * 32];
        last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(a.C - 1);
        if (last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      *sflag = last;
    }
    __syncthreads();
    if (!*sflag || col >= n_cols) continue;
    const float *ip = part_base + ((size_t)a.item * cmax * NC + col) * MK_ATTN_PSTRIDE;
    float mx = -1e30f, ls = 0.f, os[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto merge = [&](auto load8) {
      constexpr int CB = 8;  // chunks in flight
      for (int c0 = 0; c0 < a.C; c0 += CB) {
        float2 ml[CB], ov[CB][4];
#pragma unroll
        for (int j = 0; j < CB; j++)
          if (c0 + j < a.C) {
            const float *pp = ip + (size_t)(c0 + j) * NC * MK_ATTN_PSTRIDE;
            ml[j] = load8(pp + D);
#pragma unroll
            for (int d = 0; d < 4; d++) ov[j][d] = load8(pp + md + 2 * d);
          }
#pragma unroll
        for (int j = 0; j < CB; j++)
          if (c0 + j < a.C) {
            const float mn = fmaxf(mx, ml[j].x);
            const float sa = __builtin_amdgcn_exp2f(mx - mn), sb = __builtin_amdgcn_exp2f(ml[j].x - mn);
            ls = ls * sa + ml[j].y * sb;
#pragma unroll
            for (int d = 0; d < 4; d++) {
              os[2 * d] = os[2 * d] * sa + ov[j][d].x * sb;
              os[2 * d + 1] = os[2 * d + 1] * sa + ov[j][d].y * sb;
            }
            mx = mn;
          }
      }
    };
    if (local) merge([](const float *q) { return *(const float2 *)q; });
    else
      merge([](const float *q) {
        const unsigned long long v = ldc_u64(q);
        return make_float2(__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32)));
      });
    emit(os, ls);
  }
  c.wrote_through = true;  // (as in stage_attn)
}

// Greedy sampling, stage 1: every workgroup scans a contiguous slice of each token's logits and keeps
// (max, lowest index attaining it).  Reference task: tasks/mi300/argmax_mi300.cuh:78-127.
//
// Bound by round trips: a slice is a few hundred bytes.  Sixteen lanes take a token, sixteen bytes each, and every token's slice is requested
// before the first is looked at; the results leave as whole lines, so that no cache is written back.  A wavefront per token with four tokens
// in flight, a result at a time: 64 tokens of 32768 logits 16.3 -> 7.0 us, 4 tokens 8.4 -> 4.3, with the second stage 23 -> 11.5 and 12.3 -> 7.9.
template <typename E, int MAXM>
__device__ __forceinline__ void stage_argmax_partial(CStage &st, Ctx &c, const MkRuntime &rt, int M, char *smem) {
  constexpr int CH = 16 / sizeof(E);                          // logits of a piece of sixteen bytes
  constexpr int RB = (MAXM + 15) / 16, JB = 5;                // tokens of a sixteen-lane group, pieces of a lane in flight
  const int tid = c.tid, lane = tid & 63, l16 = tid & 15, g16 = tid >> 4, n = st.n;
  float *sv = (float *)smem;  // [MAXM] values, [MAXM] indices
  int *si = (int *)smem + MAXM;
  barrier_wait(c);
  // One token only: a wavefront takes the slice, a dword a lane.  By sixteen lanes the fixed-shape kernel of one token was 15 us a pass slower with
  // 151936 logits (2.991 -> 2.976 ms a token, 36 layers; before that form 2.969), more than the stage takes: it moves the register allocation of the
  // linears.  The kernels of the other stage sets do not care: 64 tokens with 32768 logits, by sixteen lanes / by a wavefront, suborax-8b 43.73 / 43.68 ms,
  // dodonex-8b 47.96 / 47.91, bukatar-8b 33.56 / 33.50, vizonex-8b 33.34 / 33.41 (qwen3-8b 41.86 / 41.78).
  if constexpr (MAXM == 1 && sizeof(E) == 2) {
    const int per = ((n + c.G - 1) / c.G + 1) & ~1, c0 = c.vid * per, c1 = min(n, c0 + per), nd = (c1 - c0 + 1) / 2;
    if (tid < 64) {
      constexpr int NDW = 5;
      uint32_t w[NDW];
      float b1 = -INFINITY;
      int i1 = 0x7fffffff;
#pragma unroll
      for (int j = 0; j < NDW; j++)
        if (j * 64 + lane < nd) w[j] = ldc_u32((const uint16_t *)st.in + c0 + 2 * (j * 64 + lane));
      auto consider = [&](uint32_t u, int i) {
        const float v0 = bf_lo(u), v1 = bf_hi(u);
        if (v0 > b1) {
          b1 = v0;
          i1 = i;
        }
        if (i + 1 < c1 && v1 > b1) {
          b1 = v1;
          i1 = i + 1;
        }
      };
#pragma unroll
      for (int j = 0; j < NDW; j++)
        if (j * 64 + lane < nd) consider(w[j], c0 + 2 * (j * 64 + lane));
      for (int d = NDW * 64 + lane; d < nd; d += 64) consider(ldc_u32((const uint16_t *)st.in + c0 + 2 * d), c0 + 2 * d);
      wave_argmax(b1, i1);
      if (lane == 0) {
        const int at = c.vid * rt.max_tokens;
        stc_f32((rt.argmax_pv ? rt.argmax_pv : (float *)st.aux0) + at, b1);
        __hip_atomic_store((rt.argmax_pv ? rt.argmax_pi : (int *)st.aux1) + at, i1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    c.wrote_through = true;
    return;
  }
  c.wrote_through = true;
  float best[RB];
  int bi[RB];
#pragma unroll
  for (int r = 0; r < RB; r++) {
    best[r] = -INFINITY;
    bi[r] = 0x7fffffff;
  }
  auto value = [](const u32x4 &w, int e) -> float {
    if constexpr (sizeof(E) == 2) return (e & 1) ? bf_hi(w[e >> 1]) : bf_lo(w[e >> 1]);
    else return __uint_as_float(w[e]);
  };
  if ((st.ld_in * sizeof(E)) % 16 == 0 && ((unsigned long long)st.in & 15) == 0) {  // (a row's last piece then ends inside the row's stride)
    const int np = (n + CH - 1) / CH, per = (np + c.G - 1) / c.G, p0 = min(c.vid * per, np), p1 = min(p0 + per, np);
    const auto rows = dev_rows(st.in);
    for (int q0 = 0; q0 < per; q0 += 16 * JB) {
      u32x4 w[RB][JB];
#pragma unroll
      for (int r = 0; r < RB; r++)
        if (r * 16 < M) {
#pragma unroll
          for (int j = 0; j < JB; j++)
            if (q0 + j * 16 < per) w[r][j] = ldc_16B(rows, min(r * 16 + g16, M - 1) * st.ld_in * (int)sizeof(E) + 16 * min(p0 + q0 + j * 16 + l16, np - 1));
        }
#pragma unroll
      for (int r = 0; r < RB; r++)
        if (r * 16 < M) {
#pragma unroll
          for (int j = 0; j < JB; j++)
            if (q0 + j * 16 < per) {
              const int p = p0 + q0 + j * 16 + l16, end = p < p1 ? n : 0;
#pragma unroll
              for (int e = 0; e < CH; e++) {
                const float v = value(w[r][j], e);
                if (p * CH + e < end && v > best[r]) {
                  best[r] = v;
                  bi[r] = p * CH + e;
                }
              }
            }
        }
    }
  } else {
    const int per = (n + c.G - 1) / c.G, c0 = c.vid * per, c1 = min(n, c0 + per);
#pragma unroll
    for (int r = 0; r < RB; r++) {
      if (r * 16 + g16 >= M) break;
      const E *row = (const E *)st.in + (size_t)(r * 16 + g16) * st.ld_in;
      for (int i = c0 + l16; i < c1; i += 16) {
        float v;
        if constexpr (sizeof(E) == 2) v = bf2f(ldc_u16((const uint16_t *)row + i));
        else v = ldc_f32((const float *)row + i);
        if (v > best[r]) {
          best[r] = v;
          bi[r] = i;
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RB; r++)
    if (r * 16 < M) {
      group16_argmax(best[r], bi[r]);
      if (l16 == 0 && r * 16 + g16 < M) {
        sv[r * 16 + g16] = best[r];
        si[r * 16 + g16] = bi[r];
      }
    }
  __syncthreads();
  if (tid < M) {  // [workgroup][token]
    const int at = c.vid * rt.max_tokens + tid;
    stc_f32((rt.argmax_pv ? rt.argmax_pv : (float *)st.aux0) + at, sv[tid]);
    __hip_atomic_store((rt.argmax_pv ? rt.argmax_pi : (int *)st.aux1) + at, si[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Greedy sampling, stage 2: one wavefront per token reduces the per-workgroup partials.
// Reference task: tasks/mi300/argmax_mi300.cuh:129-158.
__device__ __forceinline__ void stage_argmax_reduce(CStage &st, Ctx &c, const MkRuntime &rt, int M) {
  barrier_wait(c);
  c.wrote_through = true;
  const float *pv = rt.argmax_pv ? rt.argmax_pv : (const float *)st.aux0;
  const int *pi = rt.argmax_pv ? rt.argmax_pi : (const int *)st.aux1;
  const int lane = c.tid & 63, wave = __builtin_amdgcn_readfirstlane(c.tid >> 6);
  for (int t = c.vid * MK_WAVES + wave; t < M; t += c.G * MK_WAVES) {
    float best = -INFINITY;
    int bi = 0x7fffffff;
    for (int i0 = 0; i0 < c.G; i0 += 256) {
      float v[4];
      int ix[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int at = min(i0 + q * 64 + lane, c.G - 1) * rt.max_tokens + t;
        v[q] = ldc_f32(pv + at);
        ix[q] = ldc_i32(pi + at);
      }
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (v[q] > best || (v[q] == best && ix[q] < bi)) {
          best = v[q];
          bi = ix[q];
        }
    }
    wave_argmax(best, bi);
    if (lane == 0) __hip_atomic_store((long long *)st.out + t, (long long)bi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ----------------------------------------------------------------------------- the kernel
// One pass over the stage program for the M tokens of this iteration.
// ----------------------------------------------------------------------------- prompt-lookup speculative decoding
// A decoding request of a speculating graph brings n = 1 + (up to spec_len) rows into an iteration (the scheduler sizes
// the group): row 0 is its newest token at position s, rows 1.. are guesses -- the tokens that followed the EARLIEST
// earlier occurrence of its last N tokens (reference tasks find_ngram_partial_kernel / find_ngram_global_kernel,
// tasks/speculative_decoding/prompt_lookup.cuh:22-140, called with input_token_num = step + 1 and step,
// src/kernel/task_register.cc:1713-1752).  All rows run through the model as a chunk of the same request (causal
// attention inside the chunk, K/V appended at s .. s + n - 1); the verify stage then keeps the sampled token of row 0
// and one more for every guess in front that the model agrees with (target_verify_greedy_kernel,
// tasks/speculative_decoding/target_verify.cuh:21-62), and the next scheduler step advances the request by that many
// positions.  K/V rows of rejected guesses are rewritten before anything reads them.  These three stages are plain
// integer work on a few kilobytes; they are kept out of line so that the stage loop's register allocation does not see
// them.
//
// The search space of a request with T = s + 1 known tokens is idx in [0, T - N); position idx belongs to task
// (idx / 128) % P, as in the reference (128 threads per task, P tasks round-robin).  A match compares the real tokens
// idx .. idx + N - 1; the reference compares against a shared-memory window whose last N - 1 entries it leaves unset
// when they lie at or beyond T - N (prompt_lookup.cuh:62-72), so for the few idx > T - 2 N it reads unset memory.
__device__ __attribute__((noinline)) void mk_ngram_partial(int stage, const MkRuntime *rtp, int vid, int G, int *lds) {
  const MkStage *stp = rtp->stages + stage;
  const int P = stp->n, N = stp->k, ld = stp->ld_out;
  long long *part = (long long *)stp->out;
  const int R = rtp->max_requests, tid = threadIdx.x;
  for (int u = vid; u < R * P; u += G) {
    const int slot = u / P, k = u - slot * P;
    const int q0 = ldc_i32(&rtp->qo_indptr[slot]), n = ldc_i32(&rtp->qo_indptr[slot + 1]) - q0;
    const int req = ldc_i32(&rtp->request_ids[slot]);
    __syncthreads();
    if (tid == 0) lds[0] = 0x7fffffff;
    __syncthreads();
    if (req >= 0 && n > 1) {
      const int s = ldc_i32(&rtp->tok_pos[q0]);
      if (s >= rtp->prompt_lengths[req]) {  // decoding
        const long long *tok = rtp->tokens + (long long)req * rtp->max_seq;
        const int T = s + 1, total = T - N;
        for (int it = tid >> 7;; it += 2) {  // the reference's 128-thread block, two of its rounds at a time
          const long long base = ((long long)it * P + k) * 128;
          if (base >= total) break;
          const int idx = (int)base + (tid & 127);
          if (idx < total) {
            bool eq = true;
            for (int i = 0; i < N; i++) eq = eq && ldc_u64(&tok[idx + i]) == ldc_u64(&tok[T - N + i]);
            if (eq) {
              atomicMin(&lds[0], idx);
              break;  // this thread's later rounds only hold larger positions
            }
          }
        }
      }
    }
    __syncthreads();
    if (tid == 0) {
      const int m = lds[0];
      stc_u64(part + (size_t)slot * ld + k, m == 0x7fffffff ? 0x7fffffffffffffffull : (unsigned long long)m);
    }
  }
}

__device__ __attribute__((noinline)) void mk_ngram_global(int stage, const MkRuntime *rtp, int vid, int G, int *lds) {
  const MkStage *stp = rtp->stages + stage;
  const int P = stp->n, N = stp->k, ld = stp->ld_in;
  const long long *part = (const long long *)stp->in;
  long long *spec = (long long *)stp->out;
  const int R = rtp->max_requests, tid = threadIdx.x;
  for (int slot = vid; slot < R; slot += G) {
    const int q0 = ldc_i32(&rtp->qo_indptr[slot]), n = ldc_i32(&rtp->qo_indptr[slot + 1]) - q0;
    const int req = ldc_i32(&rtp->request_ids[slot]);
    if (req < 0 || n <= 0) continue;  // (uniform)
    const int s = ldc_i32(&rtp->tok_pos[q0]);
    const bool guess = n > 1 && s >= rtp->prompt_lengths[req];
    __syncthreads();
    if (tid == 0) lds[0] = 0x7fffffff;
    __syncthreads();
    if (guess) {
      for (int k = tid; k < P; k += MK_THREADS) {
        const unsigned long long v = ldc_u64(part + (size_t)slot * ld + k);
        if (v < 0x7fffffffull) atomicMin(&lds[0], (int)v);
      }
    }
    __syncthreads();
    const int first = lds[0];
    const long long *tok = rtp->tokens + (long long)req * rtp->max_seq;
    for (int j = tid; j < n; j += MK_THREADS) {
      long long v;
      if (!guess || j == 0) {
        v = (long long)ldc_u64(&rtp->input_tokens[q0 + j]);  // the scheduler's token (prompt chunk, or the newest token)
      } else {
        const long long ci = (long long)first + N + (j - 1);
        v = (first != 0x7fffffff && ci <= s) ? (long long)ldc_u64(&tok[ci]) : -1;
      }
      stc_u64(spec + q0 + j, (unsigned long long)v);
    }
  }
}

__device__ __attribute__((noinline)) void mk_verify_greedy(int stage, const MkRuntime *rtp, int vid, int G) {
  const MkStage *stp = rtp->stages + stage;
  const long long *spec = (const long long *)stp->in, *target = (const long long *)stp->aux0;
  const int R = rtp->max_requests;
  for (int slot = vid * MK_THREADS + threadIdx.x; slot < R; slot += G * MK_THREADS) {
    const int q0 = ldc_i32(&rtp->qo_indptr[slot]), n = ldc_i32(&rtp->qo_indptr[slot + 1]) - q0;
    const int req = ldc_i32(&rtp->request_ids[slot]);
    if (req < 0 || n <= 0) continue;
    int nc = n;
    if (ldc_i32(&rtp->tok_pos[q0]) >= rtp->prompt_lengths[req]) {
      // token j of this iteration is what the model sampled on row j; it counts while every guess before it was right
      // (guess j + 1 is the input of row j + 1) and nothing before it ended the request
      nc = 1;
      for (int j = 0; j + 1 < n; j++) {
        const long long tj = (long long)ldc_u64(&target[q0 + j]);
        if (tj == rtp->eos_token_id || (long long)ldc_u64(&spec[q0 + j + 1]) != tj) break;
        nc = j + 2;
      }
    }
    stc_i32(&rtp->num_new_tokens[req], nc);
    if (slot == 0 && stp->out) stc_u64(stp->out, (unsigned long long)nc);
  }
}

#if MK_PAIR
#include "mk_group.hip"
#endif
#if defined(MK_KERNEL_FLEX) || defined(MK_KERNEL_FLEX_PAIR) || defined(MK_KERNEL_FLEX_M1) || defined(MK_KERNEL_FLEX_F32) || MK_HAVE_MIX
#include "mk_flex.hip"
#if MK_HAVE_MIX
#include "mk_mix.hip"
#endif
#if MK_HAVE_HYB
#include "mk_hybrid.hip"
#endif
#if MK_HAVE_DUAL
#include "mk_dual.hip"
#endif
#define MK_HAVE_FLEX 1
#else
#define MK_HAVE_FLEX 0
#endif

// The stage set of an instantiation: the fixed-shape stages (E = void), or the flex stages for E-typed activations.
// Several portions inside prompts as one iteration (MK_PAIR): see MkPairEntry.  M1: rows of the first one; sh_rows: of all, in LDS; tok: the tokens of the
// first one and, behind them, of the one that runs beside it (c.sh_tok); any_single: in some portion every request brings one row.
template <int MAXM, typename E>
__device__ __forceinline__ void run_stage_program(const MkRuntime &rt, const MkRuntime *rtp, Ctx &c, const int M1, const int portions, const bool any_single, const int *sh_rows, int *tok,
                                                  const int n_stages, char *smem) {
    constexpr bool FX = !std::is_void<E>::value;
    constexpr bool F32 = std::is_same<E, float>::value;
    int M = M1;
    bool single = M == 1;  // every request of the iteration brings one token
    auto one_each = [&]() {
      if constexpr (FX && MAXM > 1) {
        const int lane = threadIdx.x & 63;
        single = __all(lane >= M || c.sh_tok[2 * MK_MAX_TOKENS + lane] == lane);
      }
    };
    one_each();
#if MK_PAIR
    int sum_S = 0, prep_S = 0;  // what the last linear for all portions left to the stage behind it; what such a one left to the last stage that prepares rows
    bool all_through = true, together = false;  // together: the last linear ran for all portions
    int again = 1, held = 1, shown = 0;  // the portion that entries for the second one and those behind it run for; whose tokens lie behind the first one's; c.sh_tok's
    for (int e = 0; e < rt.pair_n && !c.dead; e++) {
      const unsigned ent = (unsigned)__builtin_amdgcn_readfirstlane((int)((const __attribute__((address_space(4))) unsigned *)(unsigned long long)rt.pair_prog)[e]);
      const int s = (int)(ent & MK_PAIR_STAGE);
      if (ent & MK_PAIR_ACQUIRE) {
        barrier_wait(c);
        if (threadIdx.x == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        __syncthreads();
        continue;
      }
      const int portion = ent & MK_PAIR_SECOND ? again : 0;
      const bool behind = again + 1 < portions;  // another portion comes behind this one
      const bool on = (ent & MK_PAIR_ON) && (!(ent & MK_PAIR_SECOND) || behind), release = (ent & MK_PAIR_RELEASE) && (!(ent & MK_PAIR_SECOND) || behind);
      auto turn = [&]() {  // where the last entry of a portion has run: on to the next portion's
        if (ent & MK_PAIR_LOOP) {
          if (behind) {
            again++;
            e -= 1 + (int)(ent >> MK_PAIR_BACK_SHIFT);
          } else {
            again = 1;
          }
        }
      };
      // (the last portion's run of a stage that nobody has waited behind yet posts the arrival for all of them; not before everybody has arrived in front: the
      // barrier counts arrivals, not workgroups)
#define MK_LEAVE_OUT { if ((ent & MK_PAIR_ON) && !on) { barrier_wait(c); c.rows_ahead = 0; c.wrote_through = all_through; all_through = true; barrier_arrive(c); } turn(); continue; }
      c.portion = portion;
      M = __builtin_amdgcn_readfirstlane(sh_rows[portion]);
#if MK_HAVE_MIX
      // (a workgroup that none of a portion's rows are dealt to need not look at the stage; rows without a summand may be dealt in parts)
      if ((ent & MK_PAIR_ON) && mk_portion_stages(rt, 0)[s].op == MK_OP_MX_PRENORM && mk_portion_stages(rt, 0)[s].in && row_item(c) >= M) {
        c.defer_S = 0;
        if (on) c.rows_ahead = mk_rows_ahead(c.rows_ahead + M, c.G);
        MK_LEAVE_OUT;
      }
#endif
      if (portion != shown) {
        mk_hold_portion(portion, held, [&]() { mk_portion_rows(rt, tok + 4 * MK_MAX_TOKENS, (int)threadIdx.x, M, portion); }, []() { __syncthreads(); });
        c.sh_tok = portion ? tok + 4 * MK_MAX_TOKENS : tok;
        shown = portion;
        one_each();
      }
      if (ent & MK_PAIR_AGAIN) {
        c.defer_S = sum_S;
        c.defer_part = rt.group_part + (size_t)portion * MK_MAX_TOKENS * c.defer_n;
        CStage &sum = mk_portion_stages(rt, portion)[c.defer_stage];
        c.defer_res = sum.flags & MK_F_RES ? sum.res : nullptr;
      }
      CStage &st = mk_portion_stages(rt, portion)[s];
#else
    for (int s = 0; s < (MAXM == 1 ? rt.num_stages : n_stages) && !c.dead; s++) {
      CStage &st = ((CStage *)(unsigned long long)rt.stages)[s];
#endif
      const int op = st.op, flags = st.flags;
      // (a handle that holds only the matrix-core copies of its weights runs every linear in a matrix-core form, which
      // reads normalised rows from the NORM stage's output: that stage then runs for one and two tokens as well)
#if MK_PAIR
      // (a portion whose rows nobody prepares leaves its sum to the attention, which comes behind other portions' preparation)
      if (FX && op == MK_OP_LINEAR) {
        c.keeps_sum = mk_keeps_sum(single, s + 1 < rt.num_stages ? (&st)[1].op : 0);
        together = ent & MK_PAIR_BOTH;
      }
      if (FX && op == MK_OP_FX_PREP) prep_S = together ? c.defer_S : 0;
      if (FX && op == MK_OP_FX_ATTN && (ent & MK_PAIR_ON) && single) {
        c.defer_S = prep_S;
        c.defer_part = rt.group_part + (size_t)portion * MK_MAX_TOKENS * c.defer_n;
      }
#else
#define MK_LEAVE_OUT continue
#endif
      const bool packed_only = MAXM > 1 && rt.packed_only;
      if ((flags & MK_F_ONLY_MULTI) && M == 1 && !(packed_only && (op == MK_OP_NORM || (FX && (op == MK_OP_FX_ADDNORM || op == MK_OP_MX_PRENORM))))) MK_LEAVE_OUT;
      if (FX && op == MK_OP_FX_PREP && single) MK_LEAVE_OUT;
#if MK_HAVE_DUAL
      if (op == MK_OP_DU_CONV && (flags & MK_F_PORTIONS) && (MAXM == 1 || single)) MK_LEAVE_OUT;
#endif
#if MK_HAVE_MIX
      if ((op == MK_OP_MX_LATENT_MERGE || op == MK_OP_MX_DELTA_OUT) && !c.mx_split) MK_LEAVE_OUT;
#endif
      if ((flags & MK_F_ONLY_MULTI) && op == MK_OP_NORM && s + 1 < rt.num_stages && !packed_only) {
        // the few-token linear normalises its rows itself
        CStage &nx = (&st)[1];
        if (nx.op == MK_OP_LINEAR && (nx.flags & MK_F_NORM) && nx.in == st.in && linear_small_ok(nx, c, M)) MK_LEAVE_OUT;
      }
      // Lane offsets that stages derive from the thread index would otherwise be computed once, ahead of all stages, and wait in scratch
      // for the stage that wants them, which then starts with a chain of scratch loads.  Scratch per lane in the kernels of several tokens: 480 -> 0
      // bytes (fixed-shape stages), 640 -> 80 (flex; declared, no instruction uses it), 1568 -> 0 (mix), 1648 -> 0 (hybrid), 2320 -> 608 (dual; 752
      // by now, 498 registers spilled); vizonex-8b at 64 streams 95.5 -> 85.4 ms, bukatar-8b 57.0 -> 52.5, suborax-8b serving 135 -> 131.
      c.tid = threadIdx.x;
      asm volatile("" : "+v"(c.tid));
      __builtin_assume(c.tid >= 0 && c.tid < MK_THREADS);
#if MK_PAIR
      GroupTasks tasks;
      if constexpr (!FX) {
        if (op == MK_OP_ATTN && (ent & MK_PAIR_BOTH)) {
          if (!(st.num_q_heads == 4 * st.num_kv_heads   ? attn_group_tasks<4>(st, c, rt, portions, sh_rows, tasks)
                : st.num_q_heads == 8 * st.num_kv_heads ? attn_group_tasks<8>(st, c, rt, portions, sh_rows, tasks)
                                                        : false))
            continue;  // (portion by portion: the entries that follow)
          e += (int)(ent >> MK_PAIR_BACK_SHIFT);
        }
      }
#if MK_HAVE_FLEX
      FxGroupRows fx_tasks;
      if constexpr (FX) {
        if ((ent & MK_PAIR_BOTH) && (op == MK_OP_FX_PREP || op == MK_OP_FX_ATTN)) {
          if (any_single || (op == MK_OP_FX_ATTN && !fx_attn_group_rows(st, c, rt, portions, sh_rows, fx_tasks))) continue;  // (as above)
          e += (int)(ent >> MK_PAIR_BACK_SHIFT);
        }
      }
#endif
#endif
      c.st = &st;
      const long long t_in = (long long)wall_clock64();
      switch (op) {
#if MK_HAVE_FLEX
        case MK_OP_FX_EMBED: if constexpr (FX) stage_fx_embed<E>(st, c, rt, M); break;
        case MK_OP_FX_ADDNORM:
#if MK_PAIR
          if (ent & MK_PAIR_BOTH) {
            if constexpr (FX) stage_fx_addnorm_group<E>(st, c, rt, s, portions, sh_rows, smem);
            break;
          }
#endif
          if constexpr (FX) stage_fx_addnorm<E>(st, c, M, smem);
          break;
        case MK_OP_FX_PREP:
#if MK_PAIR
          if (ent & MK_PAIR_BOTH) {
            if constexpr (FX) stage_fx_prep_group<E>(c, rt, s, portions, sh_rows, smem);
            break;
          }
#endif
          if constexpr (FX) stage_fx_prep<E>(st, c, rt, M, smem);
          break;
        case MK_OP_FX_ATTN:
#if MK_PAIR
          if (ent & MK_PAIR_BOTH) {
            if constexpr (FX) stage_fx_attn_group<E>(st, c, rt, s, portions, sh_rows, fx_tasks, smem);
            break;
          }
#endif
          if constexpr (FX) stage_fx_attn<E>(st, c, rt, M, MAXM == 1 || single, smem);
          break;
        case MK_OP_LINEAR_F32:
          if constexpr (F32) stage_fx_linear_f32(st, c, M, smem);
          break;
        case MK_OP_FX_ARGMAX_F32: if constexpr (F32) stage_argmax_partial<float, MAXM>(st, c, rt, M, smem); break;
#endif
#if MK_HAVE_MIX
        case MK_OP_MX_PRENORM: stage_mx_prenorm<E>(st, c, M, MAXM == 1 || single, smem); break;
#if !MK_HAVE_DUAL
        case MK_OP_MX_LATENT_PREP: stage_mx_latent_prep<E>(st, c, rt, M); break;
        case MK_OP_MX_LATENT_ATTN: stage_mx_latent_attn<E>(st, c, rt, M, smem); break;
        case MK_OP_MX_LATENT_MERGE: stage_mx_latent_merge<E>(st, c, rt, M); break;
        case MK_OP_MX_DECAY: stage_mx_head_linear_t<E, 1, MX_DECAY, false>(st, c, M, smem); break;
        case MK_OP_MX_DELTA: stage_mx_delta<E>(st, c, rt, M, MAXM == 1 || single, smem); break;
        case MK_OP_MX_DELTA_OUT: stage_mx_delta_out<E>(st, c, M); break;
#endif
        case MK_OP_MX_HEAD_LINEAR: stage_mx_head_linear<E, MAXM>(st, c, M, smem); break;
#endif
#if MK_HAVE_HYB
#if MK_HAVE_DUAL
        case MK_OP_DU_CONV: stage_du_conv<E>(st, c, M); break;
        case MK_OP_DU_SCAN: stage_du_scan<E>(st, c, rt, M, MAXM == 1 || single, smem); break;
#else
        case MK_OP_HY_CONV: stage_hy_conv<E>(st, c, rt, M); break;
        case MK_OP_HY_STEP: stage_mx_head_linear_t<E, 1, MX_STEP, false>(st, c, M, smem); break;
        case MK_OP_HY_SCAN: stage_hy_scan<E>(st, c, rt, M, MAXM == 1 || single); break;
#endif
        case MK_OP_HY_ROUTE: stage_hy_route(st, c, M, smem); break;
        case MK_OP_HY_EXPERTS: stage_hy_experts<E, MAXM>(st, c, M, smem); break;
#endif
        case MK_OP_EMBED: if constexpr (!FX) stage_embed(st, c, rt, M); break;
        case MK_OP_NORM:
#if MK_PAIR
          if (ent & MK_PAIR_BOTH) {
            if constexpr (!FX) stage_norm_group(st, c, rt, s, portions, sh_rows, smem);
            break;
          }
#endif
          if constexpr (!FX) stage_norm(st, c, M, smem);
          break;
        case MK_OP_LINEAR:
          if constexpr (F32) barrier_wait(c);
#if MK_PAIR
          else if (ent & MK_PAIR_BOTH) {
            stage_linear_group(st, c, rt, s, portions, sh_rows, smem);
            sum_S = c.defer_S;
          }
#endif
          else if constexpr (MAXM == 1) stage_linear_m1<true, FX>(st, c, smem);
#if !MK_PAIR  // (portions in pairs have three rows or more)
          else if (M == 1 && !(packed_only && st.wpack)) stage_linear_m1<false, FX>(st, c, smem);
          else if (linear_small_ok(st, c, M) && !(packed_only && st.wpack)) {
            if (M <= 2) stage_linear_small_dispatch<2>(st, c, M, smem);
            else if (M <= 4) stage_linear_small_dispatch<4>(st, c, M, smem);
            else stage_linear_small_dispatch<8>(st, c, M, smem);
          }
#endif
          else {
            const int wt = (((flags & MK_F_SILU) ? st.n / 2 : st.n) + 15) / 16;  // output tiles of the stage
            const bool narrow = ((wt + c.G - 1) / c.G) * ((flags & MK_F_SILU) ? 2 : 1) <= 2;
            const TilePlan plan = linear_tiles_plan(st, c);
            const XresPlan xp = linear_xres_plan(st, c);
            if (xp.S >= 1 && (M > MK_TUNE_SMALL_MAX || packed_only)) {
              // as many token tiles as the rows need: rows behind the last token are staged, multiplied and left to the next stage like the others
              // (4 tokens with one tile instead of two, us: 6144 x 4096 11.7 -> 10.8, 4096 x 4096 9.8 -> 8.8, 4096 x 12288 19.8 -> 18.6; a third of
              // 48 instead of 64 would be another pair of instances for fewer batches)
              if (M <= 16) {
                if (xp.tpu <= 4) stage_linear_mfma_xres<1, 2>(st, c, rt, M, xp, smem);
                else stage_linear_mfma_xres<1, 3>(st, c, rt, M, xp, smem);
              } else if (M <= 32) {
                if (xp.tpu <= 4) stage_linear_mfma_xres<2, 2>(st, c, rt, M, xp, smem);
                else stage_linear_mfma_xres<2, 3>(st, c, rt, M, xp, smem);
              } else {
                if (xp.tpu <= 4) stage_linear_mfma_xres<4, 2>(st, c, rt, M, xp, smem);
                else stage_linear_mfma_xres<4, 3>(st, c, rt, M, xp, smem);
              }
            } else if (plan.S >= 1 && !(packed_only && st.wpack)) {  // (this form reads the row-major weights)
              if (M <= 16) stage_linear_mfma_tiles<1>(st, c, rt, M, plan, smem);
              else if (M <= 32) stage_linear_mfma_tiles<2>(st, c, rt, M, plan, smem);
              else if (M <= 48) stage_linear_mfma_tiles<3>(st, c, rt, M, plan, smem);
              else stage_linear_mfma_tiles<4>(st, c, rt, M, plan, smem);
            } else if (narrow) {
              if (M <= 16) stage_linear_mfma<1, 2, 2 * MK_TUNE_NBN>(st, c, M, smem);
              else if (M <= 32) stage_linear_mfma<2, 2, MK_TUNE_NBN + MK_TUNE_NBN / 2>(st, c, M, smem);
              else if (M <= 48) stage_linear_mfma<3, 2, MK_TUNE_NBN>(st, c, M, smem);
              else stage_linear_mfma<4, 2, MK_TUNE_NBN>(st, c, M, smem);
            } else {
              if (M <= 16) stage_linear_mfma<1, 6, 2>(st, c, M, smem);
              else if (M <= 32) stage_linear_mfma<2, 6, 2>(st, c, M, smem);
              else if (M <= 48) stage_linear_mfma<3, 6, 2>(st, c, M, smem);
              else stage_linear_mfma<4, 6, 2>(st, c, M, smem);
            }
          }
          break;
        case MK_OP_SILU_MUL: if constexpr (!FX) stage_silu_mul(st, c, M); break;
        case MK_OP_COPY: stage_copy(st, c, M); break;
        case MK_OP_NGRAM_PARTIAL:
        case MK_OP_NGRAM_GLOBAL:
        case MK_OP_VERIFY:
          barrier_wait(c);
          if constexpr (MAXM > 1) {  // (a graph of one token per iteration has no room for guesses)
            if (st.op == MK_OP_NGRAM_PARTIAL) mk_ngram_partial(s, rtp, c.vid, c.G, (int *)smem);
            else if (st.op == MK_OP_NGRAM_GLOBAL) mk_ngram_global(s, rtp, c.vid, c.G, (int *)smem);
            else mk_verify_greedy(s, rtp, c.vid, c.G);
            c.wrote_through = true;
          }
          break;
        case MK_OP_ATTN:
          if constexpr (FX) {
            barrier_wait(c);
#if MK_PAIR
          } else if (ent & MK_PAIR_BOTH) {
            if (st.num_q_heads == 4 * st.num_kv_heads) stage_attn_group<4>(c, rt, s, portions, sh_rows, tasks, smem);
            else stage_attn_group<8>(c, rt, s, portions, sh_rows, tasks, smem);
#endif
          } else if constexpr (MAXM == 1) {
            if (st.num_q_heads == 4 * st.num_kv_heads) stage_attn<4>(st, c, rt, M, smem);
            else if (st.num_q_heads == 8 * st.num_kv_heads) stage_attn<8>(st, c, rt, M, smem);
            else barrier_wait(c);
          } else {
            // many (token, kv head) pairs per workgroup-chunk: cached positions on the matrix cores
            const bool mf = 2 * M * st.num_kv_heads >= c.G;
            if (st.num_q_heads == 4 * st.num_kv_heads) {
              if (mf && attn_in_pairs<4>(st, c, rt, M)) stage_attn_tiles<4, true>(st, c, rt, M, smem);
              else if (mf) stage_attn_tiles<4, false>(st, c, rt, M, smem);
              else stage_attn<4>(st, c, rt, M, smem);
            } else if (st.num_q_heads == 8 * st.num_kv_heads) {
              if (mf && attn_in_pairs<8>(st, c, rt, M)) stage_attn_tiles<8, true>(st, c, rt, M, smem);
              else if (mf) stage_attn_tiles<8, false>(st, c, rt, M, smem);
              else stage_attn<8>(st, c, rt, M, smem);
            } else {
              barrier_wait(c);
            }
          }
          break;
        case MK_OP_MOE_TOPK: if constexpr (!FX) stage_moe_topk(st, c, M); break;
        case MK_OP_MOE_LINEAR: if constexpr (!FX) stage_moe_linear(st, c, M, smem); break;
        case MK_OP_MOE_COMBINE: if constexpr (!FX) stage_moe_combine(st, c, M); break;
        case MK_OP_ARGMAX_PARTIAL: if constexpr (!F32) stage_argmax_partial<uint16_t, MAXM>(st, c, rt, M, smem); break;
        case MK_OP_ARGMAX_REDUCE: stage_argmax_reduce(st, c, rt, M); break;
        default: barrier_wait(c); break;
      }
      const long long t_out = (long long)wall_clock64();
#if MK_PAIR
      if (on) {  // (as between two stages, but nobody waits for anybody)
        all_through = all_through && c.wrote_through;
        c.wrote_through = false;
        c.rows_ahead = mk_rows_ahead(c.rows_ahead + M, c.G);
        if (FX && op == MK_OP_FX_ATTN && any_single) {  // (which appends the rows of such portions itself)
          barrier_arrive(c);
          barrier_wait(c);
          if (threadIdx.x == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
          __syncthreads();
        } else {
          c.seq++;
          if (threadIdx.x == 0) c.sh_ticket[c.seq & 1] = 0;
          __syncthreads();
        }
        turn();
        continue;
      }
      c.rows_ahead = 0;
      c.wrote_through = c.wrote_through && all_through && !release;
      all_through = true;
      turn();
#endif
      barrier_arrive(c);
      if (threadIdx.x == 0 && rt.profiler) {
        // begin = this stage's inputs were complete (the previous stage's barrier seen), end = its outputs were posted
        const long long at = 1 + c.vid + (long long)c.prof_n * c.G;
        if (at + c.G < rt.profiler_cap) {
          const unsigned tag = ((unsigned)(c.seq & 0x1FFF) << 19) | ((unsigned)(c.vid & 0xFF) << 11) | ((unsigned)(st.prof_event & 0x1FF) << 2);
          rt.profiler[at] = (unsigned long long)tag | (((unsigned long long)(c.t_wait * 10) & 0xFFFFFFFFull) << 32);
          rt.profiler[at + c.G] = (unsigned long long)(tag | 1u) | (((unsigned long long)((long long)wall_clock64() * 10) & 0xFFFFFFFFull) << 32);
          c.prof_n += 2;
        }
      }
      if (threadIdx.x == 0 && rt.stage_prof) {
        long long *pr = rt.stage_prof + MK_PROF_TICKS * ((size_t)c.vid * (rt.num_stages + 1) + s);
        pr[0] = t_in;
        pr[1] = c.t_wait;
        pr[2] = t_out;
        pr[3] = (long long)wall_clock64();
#ifdef MK_TRACE
        for (int i = 0; i < 4; i++) {
          pr[4 + i] = c.mark[i];
          c.mark[i] = 0;
        }
#endif
      }
    }
}

// The kernel body, instantiated twice: MAXM = 1 for graphs that never run more than one token per iteration (every
// multi-token stage form is compiled out, so the single-token loops get the register file to themselves), and the
// general one.
template <int MAXM, typename E>
__device__ __forceinline__ void mk_kernel_body(const MkRuntime &rt, const MkRuntime *rtp, int max_iters, int run_scheduler) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int sh_bcast[4];
  __shared__ int sh_quota[10];
  __shared__ int sh_tok[MK_PAIR ? 8 : 4][MK_MAX_TOKENS];
  __shared__ int sh_ticket[3];
#if MK_PAIR
  __shared__ int sh_rows[MK_GROUP];
#endif
  // rt arrives by value in the kernel-argument segment (scalar loads); rtp is the same structure in device memory
  // for the one non-inlined function that takes its address (the scheduler step)
  Ctx c;
  c.G = gridDim.x;
  c.sync = rt.sync;
  c.xcd = xcc_id();
  c.epoch = 0;
  c.pending = false;
  c.dead = false;
  c.t_wait = 0;
  c.sh_dead = &sh_bcast[3];
  c.sh_tok = &sh_tok[0][0];
  c.sh_ticket = sh_ticket;
  c.seq = 0;
#if MK_HAVE_DUAL
  c.state_ids = rt.state_ids;
#endif
  c.prof_n = 0;
  c.st = nullptr;
  c.defer_S = 0;
#if MK_PAIR
  c.rows_ahead = 0;
  c.defer_n = 0;
  c.defer_stage = 0;
  c.portion = 0;
  c.keeps_sum = false;
#endif
  c.wrote_through = false;
  c.arrive_w0 = false;
  if (threadIdx.x == 0) {
    sh_ticket[0] = sh_ticket[1] = 0;
    sh_ticket[2] = MK_NO_LISTS;
  }
  // ---- XCD discovery: rank of this workgroup inside its die, dies in use, workgroups per die.  The dies' counters are all there is: they are
  // final once they add up to the grid.  (One counter for the whole grid beside them, awaited with acquiring loads: 8.0 us instead of 4.6 in a launch of
  // nothing else.)
  const bool from_meta = run_scheduler == MK_SCHED_FROM_META || run_scheduler == MK_SCHED_INGEST;
#if MK_PAIR
  if (from_meta && __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 1)
    for (int p = blockIdx.x; p < rt.batch_n; p += c.G) mk_open_portion(*rtp, threadIdx.x & 63, rt.batch_src, rt.batch_dst, rt.batch_len[p], rt.batch_at[p], p, rt.batch_n);
#else
  if (from_meta && blockIdx.x == 0 && __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 1) {
    // (rtp is the graph's; what belongs to this launch is in rt)
    mk_open_batch(*rtp, threadIdx.x & 63, rt.batch_src, rt.batch_dst, rt.batch_words);
  }
#endif
  if (threadIdx.x == 0) {
    MkSync *s = rt.sync;
    if (blockIdx.x == 0 && run_scheduler != MK_SCHED_RESUME) s->t_begin = (long long)wall_clock64();
    const unsigned rank = __hip_atomic_fetch_add(&s->xcd_count[c.xcd][0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned n[MK_MAX_XCD], spins = 0;
    while (true) {
      unsigned sum = 0;
      for (int i = 0; i < MK_MAX_XCD; i++) sum += n[i] = __hip_atomic_load(&s->xcd_count[i][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (sum >= (unsigned)c.G || !spin_ok(s, spins, 0xFFFF0000u)) break;
      __builtin_amdgcn_s_sleep(1);
    }
    int nx = 0, before = 0, xi = 0, mine = 0;
    for (int i = 0; i < MK_MAX_XCD; i++) {
      nx += n[i] > 0;
      if (i < c.xcd) {
        before += (int)n[i];
        xi += n[i] > 0;
      }
      if (i == c.xcd) mine = (int)n[i];
      sh_quota[i] = (int)n[i];
    }
    sh_quota[8] = xi;
    sh_quota[9] = (int)rank;
    sh_bcast[0] = before + (int)rank;
    sh_bcast[1] = nx;
    sh_bcast[2] = mine;
    sh_bcast[3] = (int)__hip_atomic_load(&s->abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  // values read back from LDS are the same in every lane: tell the compiler, so that everything derived from them
  // (tile ranges, loop bounds, guards) lives in scalar registers and branches stay scalar
  c.vid = __builtin_amdgcn_readfirstlane(sh_bcast[0]);
  c.nxcd = __builtin_amdgcn_readfirstlane(sh_bcast[1]);
  c.quota = __builtin_amdgcn_readfirstlane(sh_bcast[2]);
  c.dead = __builtin_amdgcn_readfirstlane(sh_bcast[3]) != 0;
  for (int i = 0; i < 8; i++) c.quotas[i] = (unsigned)__builtin_amdgcn_readfirstlane(sh_quota[i]);
  c.xi = __builtin_amdgcn_readfirstlane(sh_quota[8]);
  c.rank = __builtin_amdgcn_readfirstlane(sh_quota[9]);
  c.even_xcds = true;
  for (int i = 0; i < 8; i++) c.even_xcds = c.even_xcds && (c.quotas[i] == 0 || c.quotas[i] == (unsigned)c.quota);
  __syncthreads();
  if (rt.profiler) {
    c.prof_n = (unsigned)__builtin_amdgcn_readfirstlane((int)ldc_u32(&rt.profiler_count[c.vid]));
    if (c.vid == 0 && threadIdx.x == 0) rt.profiler[0] = (unsigned long long)(unsigned)c.G | (1ull << 32);
  }

  int it0 = 0;
  bool prepared = false;  // the iteration is scheduled already
  if constexpr (MAXM > 1 && !MK_PAIR) {
    prepared = run_scheduler == MK_SCHED_RESUME;
    if (prepared) {
      run_scheduler = MK_SCHED_OFFLINE;
      it0 = __builtin_amdgcn_readfirstlane(ldc_i32(&rt.sched->resume_it));
    }
  }
  for (int it = it0, more = 1; it < max_iters && !c.dead; it += more) {
    // ---- scheduler step on one thread of virtual workgroup 0, published through the barrier
    long long t_sched0 = 0, t_sched1 = 0;
    if (run_scheduler) {
      barrier_wait(c);  // the previous iteration's sampled tokens are complete
      t_sched0 = (long long)wall_clock64();
      // a handful of slots and short portions: one thread walks them; else a wavefront, one lane per slot
      const bool wave_sched = run_scheduler == MK_SCHED_OFFLINE && !prepared && (rt.max_requests > 2 || MAXM > 1 && rt.max_new_per_req > 8) && rt.spec_len == 0;
      int ntok_w = 0, portions = 1;
      if (c.vid == 0 && threadIdx.x < 64 && wave_sched) {
        ntok_w = mk_prepare_next_batch_wave(*rtp, (int *)smem, threadIdx.x, 0);
#if MK_PAIR
        bool next = __builtin_amdgcn_readfirstlane(ntok_w & MK_PAIR_NEXT);
        ntok_w &= MK_PAIR_NEXT - 1;
        for (; next && portions < rt.group && it + portions + 1 < max_iters && !rt.profiler; portions++) {  // (the launch's last iteration runs alone)
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
          next = __builtin_amdgcn_readfirstlane(mk_prepare_next_batch_wave(*rtp, (int *)smem, threadIdx.x, portions) & MK_PAIR_NEXT);
        }
        if (threadIdx.x == 0 && portions < MK_GROUP) rt.sched->group[portions] = 0;
#endif
      }
      if (from_meta) c.wrote_through = true;  // (nothing else was written in this launch)
      if (c.vid == 0 && threadIdx.x == 0 && !from_meta && !prepared) {
        int ntok;
        if (wave_sched) ntok = ntok_w;
        else if (run_scheduler == MK_SCHED_OFFLINE) ntok = mk_prepare_next_batch(*rtp, (int *)smem);
        else ntok = mk_online_next_batch(*rtp);
        if (ntok == 0) rt.sched->finished = 1;
        else rt.sched->iterations += portions;
        if (MK_PAIR) rt.sched->resume_it = ntok == 0 ? max_iters : it;
        for (int q = portions - 1; q >= 0; q--)
          if (rt.timing && rt.sched->iterations - q <= rt.timing_cap) rt.timing[rt.sched->iterations - q] = (long long)wall_clock64();
        t_sched1 = (long long)wall_clock64();
      }
      if ((from_meta || prepared) && c.vid == 0 && threadIdx.x == 0) t_sched1 = t_sched0;  // (scheduled by now, or awaited below)
      prepared = false;
      barrier_arrive(c);
    }
    barrier_wait(c);
    // one cache invalidate per iteration: whatever this CU's L1 or this die's L2 kept from earlier iterations
    // (KV rows, page tables) is dropped, so this iteration's ordinary loads of such data see what was written back
    if (threadIdx.x == 0) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      sh_bcast[0] = ldc_i32(&rt.sched->num_tokens);
      if constexpr (MAXM > 1) sh_bcast[1] = ldc_i32(&rt.sched->inner);
#if MK_PAIR
      int rows[MK_GROUP], n = 0, single = 0, bad = 0;
#pragma unroll
      for (int p = 0; p < MK_GROUP; p++) rows[p] = ldc_i32(&rt.sched->group[p]);
#pragma unroll
      for (int p = 0; p < MK_GROUP; p++) {
        if (n == p && rows[p] != 0 && p < rt.group) n = p + 1;
        sh_rows[p] = rows[p] & (MK_GROUP_SINGLE - 1);
        if (n == p + 1 && rows[p] < 0 && !bad) bad = -rows[p];
        if (n == p + 1 && rows[p] & MK_GROUP_SINGLE) single = 1;
      }
      if (from_meta) sh_bcast[0] = bad ? 0 : sh_rows[0];
      sh_bcast[1] = n | (single << 8);
      if (from_meta && c.vid == 0) {
        MkSched *sc = rt.sched;
        sc->bad_batch = bad;
        if (bad) sc->finished = 1;
        else sc->iterations += n;
        for (int q = n - 1; q >= 0 && !bad; q--)
          if (rt.timing && sc->iterations - q <= rt.timing_cap) rt.timing[sc->iterations - q] = c.t_wait;
      }
#endif
      c.sh_ticket[2] = MK_NO_LISTS;  // (expert lists are this iteration's)
    }
    __syncthreads();
    const int Mrt = __builtin_amdgcn_readfirstlane(sh_bcast[0]);
    const int M = MAXM == 1 ? (Mrt > 0 ? 1 : 0) : Mrt;
    // token metadata of this iteration, read once (it is on the critical path of every attention stage otherwise)
    if ((int)threadIdx.x < M) {
      const int t = threadIdx.x, slot = ldc_i32(&rt.tok_slot[t]);
      sh_tok[0][t] = ldc_i32(&rt.tok_pos[t]);
      sh_tok[1][t] = slot;
      sh_tok[2][t] = ldc_i32(&rt.tok_first[t]);
      sh_tok[3][t] = ldc_i32(&rt.kv_indptr[slot]);
    }
    int portions = 1;
#if MK_PAIR
    portions = M > 0 ? __builtin_amdgcn_readfirstlane(sh_bcast[1] & 255) : 0;
    more = max(portions, 1);
    if (portions > 1) mk_portion_rows(rt, sh_tok[4], (int)threadIdx.x - MK_MAX_TOKENS, sh_rows[1], 1);
#endif
    __syncthreads();
    if (threadIdx.x == 0 && rt.stage_prof && run_scheduler) {
      long long *pr = rt.stage_prof + MK_PROF_TICKS * ((size_t)c.vid * (rt.num_stages + 1) + rt.num_stages);
      pr[0] = t_sched0;
      pr[1] = t_sched1;
      pr[2] = (long long)wall_clock64();
    }
    // An iteration that only brings prompts forward ends with the last stage that writes caches or recurrent states: the logits and sampled
    // tokens of rows in front of a prompt's last token are read by nobody.  The last iteration of a launch is run whole, so that the caller finds
    // its tokens' rows in every buffer (rows behind its last token hold those of an older iteration that was run whole and had as many), and so
    // is every one that a profiler tensor is to show; where requests bring one token
    // at a time, prompts are walked as decoding walks them, all stages included.  (A prompt of 2501 tokens of qwen3-8b, 8 layers, vocabulary
    // 32768: 46.7 -> 41.1 ms; prompts of four requests of suborax-8b 1175 -> 994 us a pass, 32-bit 868 -> 676.)
    int n_stages = rt.num_stages;
    if constexpr (MAXM > 1) {
      const bool inner = MK_PAIR || __builtin_amdgcn_readfirstlane(sh_bcast[1]) != 0;
      if (!rt.profiler && (run_scheduler == MK_SCHED_INGEST || (run_scheduler == MK_SCHED_OFFLINE && inner && it + 1 < max_iters))) n_stages = rt.tail;
    }
    if (M == 0 || c.dead) break;
#if MK_PAIR
    if (portions < 2) break;  // (the iteration is left to the kernel behind this one)
    run_stage_program<MAXM, E>(rt, rtp, c, M, portions, (sh_bcast[1] >> 8) != 0, sh_rows, &sh_tok[0][0], n_stages, smem);
    c.sh_tok = &sh_tok[0][0];
    c.portion = 0;
#else
    run_stage_program<MAXM, E>(rt, rtp, c, MAXM == 1 ? 1 : M, portions, false, nullptr, nullptr, n_stages, smem);
#endif
  }
  barrier_wait(c);  // drain: nobody leaves while another workgroup may still poll
  if (rt.profiler && threadIdx.x == 0) rt.profiler_count[c.vid] = c.prof_n;
  if (c.vid == 0 && threadIdx.x == 0) {
    rt.sync->t_end = (long long)wall_clock64();
    if (rt.timing) rt.timing[0] = rt.sync->t_end;
  }
}

// build.py compiles this file once per -DMK_KERNEL_*, so that the kernels compile side by side and a build may leave out
// the ones it does not need.  The two fixed-shape instantiations share a translation unit: compiled alone, the single-token
// one gets another register assignment (about a thousand more moves and exec-mask instructions) and is 1.3 % slower.
#define MK_KERNEL_ARGS const MkRuntime rt, const MkRuntime *rtp, int max_iters, int run_scheduler
#ifdef MK_KERNEL_DENSE
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel(MK_KERNEL_ARGS) {
  mk_kernel_body<MK_MAX_TOKENS, void>(rt, rtp, max_iters, run_scheduler);
}
// graphs with max_num_batched_tokens == 1
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_m1(MK_KERNEL_ARGS) {
  mk_kernel_body<1, void>(rt, rtp, max_iters, run_scheduler);
}
#endif
// Iterations of two portions inside prompts or more, and nothing else: a launch of the offline scheduler that begins inside prompts runs this kernel up to its
// first iteration that is none, which the kernel of several tokens goes on from (MK_SCHED_RESUME).  Two kernels, as registers are allotted to
// all stages of one together: decode steps that ran here too were up to 3.7 % longer (qwen3-8b, 8 layers, rows for portions of 64, 24 requests
// 883 -> 915 us, 8 requests 807 -> 826), and with the pairs as a function beside the other stages both were slower (690 -> 1010, prompts 32.3 -> 36.0 ms).
#define MK_PAIR_KERNEL(name, E) \
  extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void name(MK_KERNEL_ARGS) { mk_kernel_body<MK_MAX_TOKENS, E>(rt, rtp, max_iters, run_scheduler); }
#ifdef MK_KERNEL_DENSE_PAIR
MK_PAIR_KERNEL(mk_persistent_kernel_pair, void)
#endif
#ifdef MK_KERNEL_FLEX_PAIR
MK_PAIR_KERNEL(mk_persistent_kernel_flex_pair, uint16_t)
#endif
#ifdef MK_KERNEL_MIX_PAIR
MK_PAIR_KERNEL(mk_persistent_kernel_mix_pair, uint16_t)
#endif
#ifdef MK_KERNEL_HYB_PAIR
MK_PAIR_KERNEL(mk_persistent_kernel_hyb_pair, uint16_t)
#endif
#ifdef MK_KERNEL_DUAL_PAIR
MK_PAIR_KERNEL(mk_persistent_kernel_dual_pair, uint16_t)
#endif
#ifdef MK_KERNEL_FLEX  // graphs with flex stages (mk_flex.hip), 16-bit activations
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_flex(MK_KERNEL_ARGS) {
  mk_kernel_body<MK_MAX_TOKENS, uint16_t>(rt, rtp, max_iters, run_scheduler);
}
#endif
#ifdef MK_KERNEL_FLEX_M1
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_flex_m1(MK_KERNEL_ARGS) {
  mk_kernel_body<1, uint16_t>(rt, rtp, max_iters, run_scheduler);
}
#endif
#ifdef MK_KERNEL_MIX  // graphs with mix stages (mk_mix.hip): the flex stages and those
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_mix(MK_KERNEL_ARGS) {
  mk_kernel_body<MK_MAX_TOKENS, uint16_t>(rt, rtp, max_iters, run_scheduler);
}
#endif
#ifdef MK_KERNEL_MIX_M1
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_mix_m1(MK_KERNEL_ARGS) {
  mk_kernel_body<1, uint16_t>(rt, rtp, max_iters, run_scheduler);
}
#endif
#ifdef MK_KERNEL_MIX_F32
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_mix_f32(MK_KERNEL_ARGS) {
  mk_kernel_body<MK_MAX_TOKENS, float>(rt, rtp, max_iters, run_scheduler);
}
#endif
#ifdef MK_KERNEL_HYB  // graphs with hybrid stages (mk_hybrid.hip): the flex and mix stages and those
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_hyb(MK_KERNEL_ARGS) {
  mk_kernel_body<MK_MAX_TOKENS, uint16_t>(rt, rtp, max_iters, run_scheduler);
}
#endif
#ifdef MK_KERNEL_HYB_M1
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_hyb_m1(MK_KERNEL_ARGS) {
  mk_kernel_body<1, uint16_t>(rt, rtp, max_iters, run_scheduler);
}
#endif
#ifdef MK_KERNEL_HYB_F32
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_hyb_f32(MK_KERNEL_ARGS) {
  mk_kernel_body<MK_MAX_TOKENS, float>(rt, rtp, max_iters, run_scheduler);
}
#endif
#ifdef MK_KERNEL_DUAL  // graphs with dual stages (mk_dual.hip): those, the flex stages, norms and head linears, routing and experts
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_dual(MK_KERNEL_ARGS) {
  mk_kernel_body<MK_MAX_TOKENS, uint16_t>(rt, rtp, max_iters, run_scheduler);
}
#endif
#ifdef MK_KERNEL_DUAL_M1
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_dual_m1(MK_KERNEL_ARGS) {
  mk_kernel_body<1, uint16_t>(rt, rtp, max_iters, run_scheduler);
}
#endif
#ifdef MK_KERNEL_DUAL_F32
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_dual_f32(MK_KERNEL_ARGS) {
  mk_kernel_body<MK_MAX_TOKENS, float>(rt, rtp, max_iters, run_scheduler);
}
#endif
#ifdef MK_KERNEL_FLEX_F32  // 32-bit activations, weights and caches
extern "C" __global__ __launch_bounds__(MK_THREADS, 1) void mk_persistent_kernel_flex_f32(MK_KERNEL_ARGS) {
  mk_kernel_body<MK_MAX_TOKENS, float>(rt, rtp, max_iters, run_scheduler);
}
#endif
