// Persistent chain of block-boundary memory updates on gfx950.
//
// Reference semantics are those of the per-update kernels: the update of
// model/kvm_mixer.py:250-340 (append + merge) with the fp32 routing of
// model/kvm_fp32_routing_reference.py:24-49, the overflow-token streams of
// model/kvm_triton_mixer.py:429-446 and the Triton numeric contract of
// model/kvm_triton_mixer.py:199-211.  This kernel runs a whole batch of
// consecutive updates in one launch instead of two to four launches per
// update, because a single update of a prefill is small (one row: 512
// tokens x 512 slots) and a kernel boundary costs more than its work.
//
// Row groups.  Every row (b, kv_head) is served by a group of G workgroups
// ("members") that sit on ONE XCD.  Workgroups are dispatched round-robin
// over the XCDs (workgroup i runs on XCD i mod n, n | 8), so the members of
// group g are the workgroups x + 8 * (q * G + m), x = g mod 8, q = g / 8.
// Members share that XCD's L2, so one member's stores are visible to the
// others once they have reached L2 (s_waitcnt) if the readers load them
// with device-scope loads (sc1), which miss in the reader's L1 (a CU's L1
// is not kept coherent with other CUs' stores; group-scope sc0 loads still
// hit it).  No device-wide L2 writeback or invalidation is needed.
// A group barrier is an L2 atomic counter; every wait is bounded and sets
// an abort flag (all members then leave) instead of spinning forever.  A
// member that gives up also ORs KVM_STATUS_CHAIN_TIMEOUT into the caller's
// sticky status word, which is how the host learns that the state and the
// snapshots of this launch are incomplete.
//
// Co-residency.  A group's members wait for each other, so all of them must
// run at the same time: the launch has at most one 512-thread workgroup per
// compute unit (chain_plan), and it relies on the GPU being otherwise idle
// enough to place all of them.  Work of another stream or process that holds
// compute units for longer than the poll budget makes the waits time out;
// the result is then reported, never silently used.
//
// Work split of one update of a row in k_chain (batches with appends):
//   member m owns tokens [m * tpw, (m + 1) * tpw)  (prep, append; tpw <= 64)
//   member m owns the 16-slot blocks m, m + G, ... (their attention keys in
//                LDS; scores of every token, merge sums, refreshed rows)
// Phases, separated by group barriers (|):
//   [novelty over my slots -> | -> select, append my tokens -> |]
//   -> route over my slots, prep(my tokens of the next update) -> |
//   -> combine, lists, merge(my slots)
// Every member scores every token against its own slots only, so an update
// reads each slot row once, from LDS (a split by tokens had every member read
// every slot row from L2 for its 32 tokens, twice), and the members exchange
// one maximum per token and scan.  The next update's rows are stored before a
// member publishes its routes, so no barrier ends an update.
// Bound by latency (barriers, L2 round trips) and, at thousands of slots, by
// the merge's row traffic.  us per update: 32 rows, C 256, 256 to 2015 slots,
// 51 -> 31.5 (novelty 7, selection 1.7, route 3, lists 2.5, merge 7, three
// barriers 2 each); 16 rows of 64-wide heads, C 128, up to 849 slots, 23.3 ->
// 17.7; 8 rows, up to 1024 slots, 23.5 -> 17.4.
// The state (s_k, s_v, s_vlen) lives in the caller's arrays; snapshot u
// holds the attention rows routing reads and snapshot u + 1 receives the
// refreshed rows of every slot, as in the per-update path.

#include "kvm_device.hpp"
#include "kvm_internal.hpp"
#include "kvm_seq.hpp"

#include <algorithm>
#include <type_traits>

namespace kvm {

// Optional per-phase timestamps of k_chain_fixed (build with
// -DKVM_CHAIN_TIMING): member 0 and member G-1 of group 0 record the wall
// clock (100 MHz) at marks 0..15 of each of the first 128 phases; the host
// reads them with kvm_chain_timing_read.  Without the define the marks
// compile to nothing.
#ifdef KVM_CHAIN_TIMING
__device__ unsigned long long g_chain_ts[2][128][16];
#define KVM_TS(k)                                                                        \
  do {                                                                                   \
    if (threadIdx.x == 0 && p < 128) {                                                   \
      if (blockIdx.x == 0) g_chain_ts[0][p][k] = wall_clock64();                         \
      else if (blockIdx.x == 8 * (GM - 1)) g_chain_ts[1][p][k] = wall_clock64();          \
    }                                                                                    \
  } while (0)
// The other chains' marks: workgroup 0, update i of the launch.
#define KVM_TS_A(k)                                                                      \
  do {                                                                                   \
    if (threadIdx.x == 0 && blockIdx.x == 0 && i < 128) g_chain_ts[0][i][k] = wall_clock64(); \
  } while (0)
#else
#define KVM_TS(k) ((void)0)
#define KVM_TS_A(k) ((void)0)
#endif

namespace {

// Dynamic LDS of the appending chain: the scans' maxima, or the lists' counts in their place ...
__host__ __device__ inline int append_red_bytes(int n_tok, int own_cap) {
  int ntg = 64;
  while (ntg < n_tok) ntg <<= 1;
  const int scan = (ntg < 512 ? 512 : ntg) * 8, lists = (n_tok + 63) / 64 * own_cap;
  return ((scan > lists ? scan : lists) + 15) & ~15;
}
// ... then off / cnt [own_cap] and sorted / apos [n_tok].
__host__ __device__ inline int append_lds_bytes(int n_tok, int own_cap) {
  return append_red_bytes(n_tok, own_cap) + 4 * own_cap + 4 * n_tok;
}

// Beside the attention keys (OwnLds): room for 2144 own slots per member at
// 1024 tokens per update, 3744 at 512 (29952 slots with eight members).  32
// rows of 128, C 512, up to 18892 slots: 11.8 ms a prefill, 18.3 on the
// per-update kernels, which states past the tables run on.
constexpr int kAppendDynLds = 46 * 1024;
constexpr int kChainThreads = 512;
constexpr int kChainWaves = kChainThreads / 64;
constexpr int kChainTok = 64;        // tokens per member at most
constexpr int kCounterStride = 32;   // words between group counters (128 B)

// Group barrier, split so that independent work can run between arriving
// and waiting.  arrive: this workgroup's global stores have reached L2,
// then one L2 atomic increment.
__device__ __forceinline__ void group_arrive(unsigned *ctr) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Scalar load that misses in the scalar cache (glc) and reads L2, where the
// members' atomic increments land.  It is counted by lgkmcnt, not vmcnt, so
// a poll does not wait behind the wave's outstanding vector loads (which
// return in order): the barrier is seen as soon as the last member arrives.
__device__ __forceinline__ unsigned l2_scalar_load(const unsigned *p) {
  unsigned v;
  asm volatile("s_load_dword %0, %1, 0x0 glc\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(p) : "memory");
  return v;
}
// wait: until `target` arrivals (G per barrier), polled by wave 0.  False
// when the wait timed out or another group aborted.
__device__ __forceinline__ bool group_wait(unsigned *ctr, unsigned target, const ChainScratch &cs,
                                           int *ok_lds) {
  if (threadIdx.x < 64) {  // wave 0, wave-uniform
    int ok = 0;
    for (unsigned p = 0; p < cs.max_polls; ++p) {
      if (l2_scalar_load(ctr) >= target) {
        ok = 1;
        break;
      }
      if ((p & 255u) == 255u && l2_scalar_load(cs.abort_flag)) break;
      __builtin_amdgcn_s_sleep(1);
    }
    if (threadIdx.x == 0) {
      if (!ok) {
        __hip_atomic_store(cs.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_fetch_or(cs.status, unsigned(KVM_STATUS_CHAIN_TIMEOUT), __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_AGENT);
      }
      *ok_lds = ok;
    }
  }
  __syncthreads();
  return *ok_lds != 0;
}

// Loads of data that other members wrote during this launch: buffer loads
// with device scope (sc1), served by the XCD's L2.  Offsets at or past the
// resource's byte count read zero.
constexpr int kBufWord3 = 0x00020000;
constexpr int kScopeDevice = 16;  // cache-policy bits: sc1
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t l2_rsrc(const void *base, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0,
                                           int(bytes < 0x7fffffff ? bytes : 0x7fffffff), kBufWord3);
}
__device__ __forceinline__ uint4 l2_ld16(__amdgpu_buffer_rsrc_t r, int off) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kScopeDevice);
  return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint32_t l2_ld4(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, kScopeDevice);
}

// Route key of a (score, slot) candidate: the per-update routing kernel's
// order-preserving encoding mono(fp32 score) << 32 | (0xffffffff - slot), so
// an integer maximum picks the largest score and, among equal scores, the
// lowest slot (torch.max returns the first maximum).  0 means no candidate.
__device__ __forceinline__ uint64_t route_key(float score, int slot) {
  const uint32_t u = __float_as_uint(score);
  const uint32_t m = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  return (uint64_t(m) << 32) | uint64_t(0xffffffffu - uint32_t(slot));
}
__device__ __forceinline__ int route_key_slot(uint64_t key) {
  return key ? int(0xffffffffu - uint32_t(key)) : -1;
}

// The running first maximum (best, from -inf on, and its slot) against a
// lane's four consecutive slots from j0 on; equal scores go to the earlier
// slot.  A tree of comparisons, with independent chains per token tile, where
// all four count and none is NaN, which would stand for its neighbours ...
__device__ __forceinline__ void keep_max4(const f32x4 &a, int j0, float &best, int &slot) {
  const bool t1 = a[1] > a[0], t3 = a[3] > a[2];
  const float v01 = t1 ? a[1] : a[0], v23 = t3 ? a[3] : a[2];
  const int i01 = t1 ? 1 : 0, i23 = t3 ? 3 : 2;
  const bool th = v23 > v01;
  const float vh = th ? v23 : v01;
  const bool take = vh > best;
  best = take ? vh : best;
  slot = take ? j0 + (th ? i23 : i01) : slot;
}
// ... and slot by slot over those in [lo, hi), where a NaN never wins.
__device__ __forceinline__ void scan_max4(const f32x4 &a, int j0, int lo, int hi, float &best, int &slot) {
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const float sc = (j0 + x >= lo) && (j0 + x < hi) ? a[x] : -INFINITY;
    const bool take = sc > best;
    best = take ? sc : best;
    slot = take ? j0 + x : slot;
  }
}
// Whether a block of 16 slots from jb on needs the scan: slots outside
// [lo, hi), or a NaN key (a: the first operand of the block's keys; a key row
// is a LayerNorm's output, NaN in every feature or in none).  Wave-uniform.
__device__ __forceinline__ bool needs_scan(const uint4 &a, int jb, int lo, int hi) {
  return jb < lo || jb + 16 > hi || __any((a.x & 0x7fffu) > 0x7f80u);
}

// LDS byte address of a __shared__ object (wave-uniform).
typedef __attribute__((address_space(3))) void lds_void;
template <typename T>
__device__ __forceinline__ uint32_t lds_addr(T *p) {
  return __builtin_amdgcn_readfirstlane(uint32_t(uintptr_t((lds_void *)(p))));
}
// 16-byte-per-lane device-scope (sc1) buffer load from L2 straight into LDS
// at M0 + 16 * lane.  Issued from inline assembly so that the compiler does
// not order later LDS reads behind it; the caller waits with s_waitcnt vmcnt.
// M0 is written inside the statement and not declared clobbered (the compiler
// rejects M0 as a clobber): this is sound only while no compiled code of the
// kernel keeps a value of its own in M0, which holds for these kernels (their
// only M0 writes are these statements; checked in the generated assembly).
__device__ __forceinline__ void dma16_l2(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen sc1 lds"
               :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(r) : "memory");
}

// The same from device memory with the non-temporal policy: raw token rows
// are read once, and streaming them keeps them from evicting the merge
// buffers the group reads back from L2 one and two updates later.
__device__ __forceinline__ void dma16_nt(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
               :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(r) : "memory");
}

// 16-byte buffer store at a 32-bit byte offset from the resource's base
// (aux: cache policy bits; kPolicyNT streams the line to memory).
constexpr int kPolicyNT = 2;
template <int AUX>
__device__ __forceinline__ void st16(__amdgpu_buffer_rsrc_t r, uint32_t off, const uint4 &v) {
  __builtin_amdgcn_raw_buffer_store_b128(u32x4{v.x, v.y, v.z, v.w}, r, int(off), 0, AUX);
}

// Waits until at most N vector memory operations of the wave are in flight.
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}

// Raw token rows are read once: non-temporal loads keep them from evicting
// the merge buffers the group reads back from L2 one and two updates later.
__device__ __forceinline__ uint4 ld_stream16(const uint16_t *p) {
  const u32x4 x = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
  return make_uint4(x[0], x[1], x[2], x[3]);
}

// Lane exchanges across 16 / 32 lanes with v_permlane{16,32}_swap (VALU,
// no LDS round trip): the value of lane l ^ 16 (l ^ 32).
__device__ __forceinline__ uint32_t xor16_lane(uint32_t x, int lane) {
  const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  return (lane & 16) ? r[0] : r[1];
}
__device__ __forceinline__ uint32_t xor32_lane(uint32_t x, int lane) {
  const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return (lane & 32) ? r[0] : r[1];
}

__device__ __forceinline__ AttnRows snap_at(const SnapRing &r, int64_t idx) {
  const int64_t o = (idx % r.ring) * r.stride;
  return AttnRows{r.k + o, r.v + o, r.cap};
}

// Raw key / value / gate of the member's tokens, D/8 lanes per token.
template <int D>
struct RawTok {
  static constexpr int IT = kChainTok * (D / 8) / kChainThreads;
  uint4 k[IT], v[IT];
  uint16_t g[IT];  // bf16 bits, converted where used (no wait at the load)
};

// Slot of a member's local slot l: the member owns 16-slot blocks m, m + G, ...
__device__ __forceinline__ int own_local_to_slot(int l, int G, int m) {
  return (((l >> 4) * G + m) << 4) | (l & 15);
}

// Own slots whose attention keys the appending chain keeps in LDS; further
// ones are read from their snapshot.
template <int D>
struct OwnLds {
  static constexpr int value = D == 128 ? 384 : 768;
};

template <int D, int G>
__global__ __launch_bounds__(kChainThreads) void k_chain(
    kvm_layer L, kvm_seq src, int n_tok, kvm_state st, SnapRing snaps, ChainList list,
    ChainScratch cs, int rows, int row0, int nrows, int tpw, int own_cap, int32_t *route_log,
    int32_t *append_log, int64_t log_stride) {
  constexpr int GL = D / 8;                 // lanes per D-wide row
  constexpr int STR = D + 8;                // LDS row stride (elements)
  constexpr int KS = D / 32;
  constexpr int RPP = kChainThreads / GL;   // rows per pass
  constexpr int IT = RawTok<D>::IT;         // passes over the member's tokens
  constexpr int OWNL = OwnLds<D>::value;
  static_assert(IT * RPP == kChainTok, "token passes");
  __shared__ __attribute__((aligned(16))) uint16_t own_k[OWNL * STR];  // attention keys of my slots
  __shared__ int wtot[kChainWaves];
  __shared__ int ok_lds;
  __shared__ float ln_w[D], ln_b[D];  // ln_s_k parameters (LDS: no wait on global loads)
  // [slot group][token] maxima of a scan (8 bytes each); in their place, the
  // lists' counts [64 tokens][own_cap], at most 64 each.  Then off / cnt
  // [own_cap], sorted and apos [n_tok] (append_lds_bytes).
  extern __shared__ __attribute__((aligned(16))) uint64_t red[];
  uint8_t *const wsc = reinterpret_cast<uint8_t *>(red);
  uint16_t *const off = reinterpret_cast<uint16_t *>(wsc + append_red_bytes(n_tok, own_cap));
  uint16_t *const cnt = off + own_cap;
  uint16_t *const sorted = cnt + own_cap;                              // tokens of my slots, slot by slot
  int16_t *const apos = reinterpret_cast<int16_t *>(sorted + n_tok);   // append position of a token or -1

  const int tid = threadIdx.x, lane = tid & 63, part = tid % GL, sub = tid / GL;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
  const int member = q % G, group = (q / G) * 8 + xcd;
  if (group >= nrows) return;
  for (int d = tid; d < D; d += kChainThreads) {
    ln_w[d] = static_cast<const float *>(L.ln_weight)[d];
    ln_b[d] = static_cast<const float *>(L.ln_bias)[d];
  }
  const int row = row0 + group;  // this launch serves rows row0 .. row0 + nrows - 1
  const int b = row / int(L.kv_heads), h = row % int(L.kv_heads);
  const int t0 = member * tpw;
  const int ntk = max(0, min(n_tok, t0 + tpw) - t0);
  const int64_t rb = int64_t(row) * n_tok;
  const int64_t buf_stride = int64_t(rows) * n_tok * D;  // elements between merge buffers
  const int rowb = n_tok * D * 2;                        // bytes of a row's tokens in one of them
  unsigned *ctr = cs.bar + group * kCounterStride;
  unsigned target = 0;
  auto arrive = [&]() __attribute__((always_inline)) {
    target += unsigned(G);
    group_arrive(ctr);
  };
  auto wait = [&]() __attribute__((always_inline)) {
    return group_wait(ctr, target, cs, &ok_lds);
  };
  uint16_t *s_k = static_cast<uint16_t *>(st.s_k);
  uint16_t *s_v = static_cast<uint16_t *>(st.s_v);
  float *s_vlen = static_cast<float *>(st.s_vlen);
  const int64_t srow = int64_t(row) * st.capacity;
  // Token rows of update i: merge keys and values in buffers 0..2 of gk / gv
  // (an update's are prepared one update ahead and read last by its merge,
  // while the next but one may already be prepared by another member);
  // prep(k) of appending updates in buffer 3 of gk (even) or gv (odd).
  auto gk_of = [&](int i) __attribute__((always_inline)) { return cs.gk + (i % 3) * buf_stride + rb * D; };
  auto gv_of = [&](int i) __attribute__((always_inline)) { return cs.gv + (i % 3) * buf_stride + rb * D; };
  auto pk_of = [&](int i) __attribute__((always_inline)) { return ((i & 1) ? cs.gv : cs.gk) + 3 * buf_stride + rb * D; };

  // Raw tokens of update i (token 0 of the chunk for idle lanes).  Prefill
  // tokens never come from a ring (src.ring == 0, checked by the host).
  const uint16_t *k_row = static_cast<const uint16_t *>(src.k) + b * src.k_sb + h * src.k_sh;
  const uint16_t *v_row = static_cast<const uint16_t *>(src.v) + b * src.v_sb + h * src.v_sh;
  const uint16_t *g_row = static_cast<const uint16_t *>(src.gate) + b * src.g_sb + h * src.g_sh;
  auto load_raw = [&](int i, RawTok<D> &rt) __attribute__((always_inline)) {
    const int64_t tb = list.tok_begin[i];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      if (it * RPP >= ntk) break;  // uniform
      const int lt = it * RPP + sub;
      const int64_t t = tb + (lt < ntk ? t0 + lt : 0);
      rt.k[it] = ld_stream16(k_row + t * src.k_st + part * 8);
      rt.v[it] = ld_stream16(v_row + t * src.v_st + part * 8);
      rt.g[it] = g_row[t * src.g_st];
    }
  };
  // prep (model/kvm_mixer.py:120-129, model/kvm_triton_mixer.py:429-446):
  // merge key / value rows of my tokens, and prep(k) when the update appends.
  auto prep = [&](int i, const RawTok<D> &rt) __attribute__((always_inline)) {
    const bool nov = list.n_append[i] > 0;
    uint16_t *gkb = gk_of(i), *gvb = gv_of(i), *pkb = pk_of(i);
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      if (it * RPP >= ntk) break;  // uniform
      const int lt = it * RPP + sub;
      float k[8], v[8];
      unpack8(rt.k[it], k);
      unpack8(rt.v[it], v);
      const float g = bf2f(rt.g[it]);
      prep_key<D>(k, part, L, ln_w, ln_b);
      float gk[8], gv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        gk[e] = L.gate_keys ? rbf(k[e] * g) : k[e];
        gv[e] = L.gate_values ? rbf(v[e] * g) : v[e];
      }
      if (lt < ntk) {
        const int64_t o = int64_t(t0 + lt) * D + part * 8;
        store8(gkb + o, gk);
        store8(gvb + o, gv);
        if (nov) store8(pkb + o, k);
      }
    }
  };

  // ---- attention keys of my slots (those of the first OWNL) into LDS.
  auto load_own = [&](const uint16_t *keys, int lo, int hi) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t kr = l2_rsrc(keys, int64_t(hi) * D * 2);
    for (int l = sub; l < min(own_cap, OWNL); l += RPP) {
      const int j = own_local_to_slot(l, G, member);
      if (j >= lo && j < hi)
        *reinterpret_cast<uint4 *>(&own_k[l * STR + part * 8]) = l2_ld16(kr, (j * D + part * 8) * 2);
    }
  };
  {
    const AttnRows a0 = snap_at(snaps, list.u0);
    load_own(a0.k + int64_t(row) * a0.cap * D, 0, list.state_before[0]);
  }
  // The scans' work split: token groups of 64 (waves tg, tg + 8, ...) x slot
  // groups (interleaved blocks of 16) over the waves.
  int ntg = 1;
  while (ntg * 64 < n_tok) ntg <<= 1;
  const int nsg = max(1, kChainWaves / ntg), sg = wave / ntg, tg0 = wave % ntg;

  // Scan of every token (rows at `tok`, prepared by all members) against my
  // slots below hi on MFMA 16x16x32 bf16, computed transposed (slot x token)
  // with the same operand roles and k-step order as the per-update routing
  // kernel, so the fp32 scores are bit-identical.  Into red[slot group][token]:
  //   NOVELTY: maximum of the bf16-rounded score, as float bits
  //            (model/kvm_mixer.py:66-68);
  //   route:   route key of the first argmax over slots [lo, hi)
  //            (model/kvm_fp32_routing_reference.py:30-34).
  // The caller has loaded bx for the wave's first token group.
  uint4 bx[4][KS];
  auto load_bx = [&](const uint16_t *tok, int tg) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t tr = l2_rsrc(tok, rowb);
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        bx[tt][ks] = l2_ld16(tr, ((tg * 64 + tt * 16 + (lane & 15)) * D + ks * 32 + (lane >> 4) * 8) * 2);
  };
  auto scan = [&](auto novelty, const uint16_t *tok, const uint16_t *keys, int lo,
                  int hi) __attribute__((always_inline)) {
    constexpr bool NOVELTY = decltype(novelty)::value;
    const __amdgpu_buffer_rsrc_t kr = l2_rsrc(keys, int64_t(hi) * D * 2);
    const int nblk = (hi + 15) >> 4;
    for (int tg = tg0; tg * 64 < n_tok; tg += kChainWaves) {
      if (tg != tg0) load_bx(tok, tg);
      float best[4];
      int bidx[4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        best[tt] = -INFINITY;
        bidx[tt] = -1;
      }
      for (int lb = sg; lb * G + member < nblk; lb += nsg) {
        const int jb = (lb * G + member) * 16;  // first slot of the block
        uint4 a[KS];
        if (lb * 16 < OWNL) {  // uniform
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
            a[ks] = *reinterpret_cast<const uint4 *>(
                &own_k[(lb * 16 + (lane & 15)) * STR + ks * 32 + (lane >> 4) * 8]);
        } else {
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
            a[ks] = l2_ld16(kr, ((jb + (lane & 15)) * D + ks * 32 + (lane >> 4) * 8) * 2);
        }
        f32x4 accs[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) accs[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int tt = 0; tt < 4; ++tt)
            accs[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[ks]), as_bf16x8(bx[tt][ks]), accs[tt], 0,
                                                               0, 0);
        const int j0 = jb + (lane >> 4) * 4;
        if constexpr (NOVELTY) {
          if (jb + 16 > hi) {  // slots past hi never count (lo is 0)
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
              for (int x = 0; x < 4; ++x) accs[tt][x] = j0 + x < hi ? accs[tt][x] : -INFINITY;
          }
#pragma unroll
          for (int tt = 0; tt < 4; ++tt) {
            // The rounding is monotone, so the maximum may be taken first.
            const f32x4 acc = accs[tt];
            best[tt] = fmaxf(best[tt], fmaxf(fmaxf(acc[0], acc[1]), fmaxf(acc[2], acc[3])));
          }
        } else if (needs_scan(a[0], jb, lo, hi)) {
#pragma unroll
          for (int tt = 0; tt < 4; ++tt) scan_max4(accs[tt], j0, lo, hi, best[tt], bidx[tt]);
        } else {
#pragma unroll
          for (int tt = 0; tt < 4; ++tt) keep_max4(accs[tt], j0, best[tt], bidx[tt]);
        }
      }
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        uint64_t *const out = &red[(sg * ntg + tg) * 64 + tt * 16 + (lane & 15)];
        if constexpr (NOVELTY) {
          float v = best[tt];
          v = fmaxf(v, __uint_as_float(xor16_lane(__float_as_uint(v), lane)));
          v = fmaxf(v, __uint_as_float(xor32_lane(__float_as_uint(v), lane)));
          if (lane < 16) *out = __float_as_uint(rbf(v));
        } else {
          uint64_t key = bidx[tt] >= 0 ? route_key(best[tt], bidx[tt]) : 0;
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            const uint32_t hi32 = uint32_t(key >> 32), lo32 = uint32_t(key);
            const uint64_t other = r == 0 ? (uint64_t(xor16_lane(hi32, lane)) << 32) | xor16_lane(lo32, lane)
                                          : (uint64_t(xor32_lane(hi32, lane)) << 32) | xor32_lane(lo32, lane);
            key = other > key ? other : key;
          }
          if (lane < 16) *out = key;
        }
      }
    }
  };

  RawTok<D> rt;
  load_raw(0, rt);
  __syncthreads();
  prep(0, rt);
  arrive();
  if (!wait()) return;

  for (int i = 0; i < list.count; ++i) {
    const int64_t u = int64_t(list.u0) + i;
    const int64_t tb = list.tok_begin[i];
    const int sb = list.state_before[i], na = list.n_append[i];
    const int s_after = sb + na;
    const int protect = min(int(L.sink_len), s_after);
    const bool more = i + 1 < list.count;
    const AttnRows cur = snap_at(snaps, u), nxt = snap_at(snaps, u + 1);
    int32_t *rlog = route_log ? route_log + u * log_stride + rb : nullptr;
    int32_t *alog = append_log ? append_log + u * log_stride + rb : nullptr;
    uint16_t *cur_k = cur.k + int64_t(row) * cur.cap * D, *cur_v = cur.v + int64_t(row) * cur.cap * D;
    KVM_TS_A(0);

    // ---- append (model/kvm_mixer.py:44-75, 231-248): the n_append least
    // novel tokens, ties to the lower index, become slots sb.. in token order.
    if (na > 0) {
      load_bx(pk_of(i), tg0);
      scan(std::true_type{}, pk_of(i), cur_k, 0, sb);
      load_bx(gk_of(i), tg0);  // the route's operands, in flight through the append
      __syncthreads();
      for (int t = tid; t < n_tok; t += kChainThreads) {
        float v = -INFINITY;
        for (int x = 0; x < nsg; ++x) v = fmaxf(v, __uint_as_float(uint32_t(red[x * ntg * 64 + t])));
        cs.nov[(rb + t) * G + member] = v;
      }
      KVM_TS_A(1);
      arrive();
      if (!wait()) return;
      KVM_TS_A(2);
      // The na tokens of smallest (novelty, token), on wave 0: the novelties
      // are bf16 values, so their order is that of 16-bit keys (-0 read as
      // +0); the largest key to take is found bit by bit with ballots, and
      // among its tokens the first ones in token order are taken.
      uint32_t *const nkey = reinterpret_cast<uint32_t *>(red);  // [16 * 64]: the maxima have been published
      {
        const __amdgpu_buffer_rsrc_t nr = l2_rsrc(cs.nov + rb * G, int64_t(n_tok) * G * 4);
        for (int t = tid; t < ntg * 64; t += kChainThreads) {
          uint4 p4[G / 4];  // past the tokens: zeros, not used
#pragma unroll
          for (int m = 0; m < G / 4; ++m) p4[m] = l2_ld16(nr, (t * G + m * 4) * 4);
          float v = -INFINITY;
#pragma unroll
          for (int m = 0; m < G / 4; ++m)
            v = fmaxf(v, fmaxf(fmaxf(__uint_as_float(p4[m].x), __uint_as_float(p4[m].y)),
                               fmaxf(__uint_as_float(p4[m].z), __uint_as_float(p4[m].w))));
          const uint32_t bits = __float_as_uint(v + 0.0f);
          const uint32_t key = ((bits & 0x80000000u) ? ~bits : (bits | 0x80000000u)) >> 16;
          nkey[t] = t < n_tok ? key : 0xffffffffu;  // above every novelty
        }
      }
      __syncthreads();
      if (wave == 0) {
        auto select = [&](auto groups) __attribute__((always_inline)) {
          constexpr int NV = decltype(groups)::value;  // tokens per lane
          uint32_t key[NV];
#pragma unroll
          for (int x = 0; x < NV; ++x) key[x] = nkey[x * 64 + lane];
          uint32_t cut = 0;
          int left = na;  // tokens to take among those that agree with cut so far
#pragma unroll
          for (int bit = 15; bit >= 0; --bit) {
            int n = 0;
#pragma unroll
            for (int x = 0; x < NV; ++x) n += __popcll(__ballot((key[x] >> bit) == (cut >> bit)));
            if (n < left) {
              left -= n;
              cut |= 1u << bit;
            }
          }
          int base = 0;
#pragma unroll
          for (int x = 0; x < NV; ++x) {
            const uint64_t tie = __ballot(key[x] == cut);
            const int before = int(__builtin_amdgcn_mbcnt_hi(
                uint32_t(tie >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(tie), 0u)));
            const bool ap = key[x] < cut || (key[x] == cut && before < left);
            left -= min(left, int(__popcll(tie)));
            const uint64_t bal = __ballot(ap);
            const int at = base + int(__builtin_amdgcn_mbcnt_hi(
                                      uint32_t(bal >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(bal), 0u)));
            base += int(__popcll(bal));
            if (x * 64 + lane < n_tok) apos[x * 64 + lane] = int16_t(ap ? at : -1);
          }
        };
        if (ntg == 1)
          select(std::integral_constant<int, 1>{});
        else if (ntg == 2)
          select(std::integral_constant<int, 2>{});
        else if (ntg == 4)
          select(std::integral_constant<int, 4>{});
        else if (ntg == 8)
          select(std::integral_constant<int, 8>{});
        else
          select(std::integral_constant<int, 16>{});
      }
      __syncthreads();
      KVM_TS_A(3);
      const __amdgpu_buffer_rsrc_t akr = l2_rsrc(L.gate_appends ? gk_of(i) : pk_of(i), rowb);
      const __amdgpu_buffer_rsrc_t avr = l2_rsrc(gv_of(i), rowb);
#pragma unroll
      for (int it = 0; it < IT; ++it) {
        const int lt = it * RPP + sub;
        const int tl = lt < ntk ? t0 + lt : 0;  // token of this lane (token 0 when idle)
        const bool valid = lt < ntk && apos[tl] >= 0;
        if (__any(valid)) {
          float k[8], v[8];
          unpack8(l2_ld16(akr, (tl * D + part * 8) * 2), k);
          if (L.gate_appends)
            unpack8(l2_ld16(avr, (tl * D + part * 8) * 2), v);
          else
            load8(v_row + (tb + tl) * src.v_st + part * 8, v);
          const float vlen = row_norm8<D>(v);
          float ka[8], va[8];
          attn_rows<D>(k, v, vlen, part, L, ln_w, ln_b, ka, va);
          if (valid) {
            const int64_t slot = sb + apos[tl];
            const int64_t so = (srow + slot) * D + part * 8;
            store8(s_k + so, k);
            store8(s_v + so, v);
            if (part == 0) s_vlen[srow + slot] = vlen;
            store8(cur_k + slot * D + part * 8, ka);
            store8(cur_v + slot * D + part * 8, va);
          }
        }
      }
      KVM_TS_A(4);
      arrive();
      // The next update's raw tokens while the group waits (loads return in
      // order: anywhere else the loads behind them would wait for memory).
      if (more) load_raw(i + 1, rt);
      if (!wait()) return;
      load_own(cur_k, sb, s_after);
      __syncthreads();
      KVM_TS_A(5);
    } else {
      load_bx(gk_of(i), tg0);
      if (more) load_raw(i + 1, rt);
    }

    // ---- route, then the next update's prep: with its rows stored before
    // this update's routes are published, no barrier ends the update.
    scan(std::false_type{}, gk_of(i), cur_k, protect, s_after);
    KVM_TS_A(6);
    if (more) prep(i + 1, rt);
    __syncthreads();
    uint2 *const part_row = cs.part + int64_t(i & 1) * rows * n_tok * G + rb * G;
    for (int t = tid; t < n_tok; t += kChainThreads) {
      uint64_t key = 0;
      for (int x = 0; x < nsg; ++x) {
        const uint64_t o = red[x * ntg * 64 + t];
        key = o > key ? o : key;
      }
      part_row[t * G + member] = make_uint2(uint32_t(key >> 32), uint32_t(key));
    }
    KVM_TS_A(7);
    arrive();
    if (!wait()) return;
    KVM_TS_A(8);

    // ---- the tokens of each of my slots, in token order: ballots rank the
    // tokens of 64, counts per 64 tokens and slot place them.
    const __amdgpu_buffer_rsrc_t pr = l2_rsrc(part_row, int64_t(n_tok) * G * 8);
    const int nvw = (n_tok + 63) >> 6;
    const int nblk = (s_after + 15) >> 4;
    const int nown = member < nblk ? ((nblk - 1 - member) / G + 1) * 16 : 0;  // my local slots in use
    for (int e = tid; e < nvw * own_cap / 4; e += kChainThreads) reinterpret_cast<uint32_t *>(wsc)[e] = 0;
    constexpr int NT = 2;  // tokens per thread (n_tok <= 1024)
    int loc[NT], rank[NT];
    uint64_t pkey[NT];
#pragma unroll
    for (int x = 0; x < NT; ++x) {
      const int t = x * kChainThreads + tid;
      pkey[x] = 0;
      if (t < n_tok)
      {
        uint4 p4[G / 2];
#pragma unroll
        for (int m = 0; m < G / 2; ++m) p4[m] = l2_ld16(pr, (t * G + 2 * m) * 8);
#pragma unroll
        for (int m = 0; m < G / 2; ++m) {
          const uint64_t a0 = (uint64_t(p4[m].x) << 32) | p4[m].y, a1 = (uint64_t(p4[m].z) << 32) | p4[m].w;
          pkey[x] = a0 > pkey[x] ? a0 : pkey[x];
          pkey[x] = a1 > pkey[x] ? a1 : pkey[x];
        }
      }
    }
    __syncthreads();  // wsc is cleared
#pragma unroll
    for (int x = 0; x < NT; ++x) {
      const int t = x * kChainThreads + tid;
      loc[x] = -1;
      if (x * kChainThreads < n_tok) {
        const int slot = route_key_slot(pkey[x]);
        const bool app = na > 0 && t < n_tok && apos[t] >= 0;
        if (t >= t0 && t < t0 + ntk) {  // each member logs its own tokens
          if (alog) alog[t] = app ? 1 : 0;
          if (rlog) rlog[t] = app ? sb + apos[t] : slot;
        }
        const bool mine = slot >= 0 && !app && (slot >> 4) % G == member;
        const int l = mine ? (((slot >> 4) / G) << 4) | (slot & 15) : 0;
        uint64_t eq = __ballot(mine);
        for (int bit = 0; (1 << bit) < own_cap; ++bit) {
          const uint64_t m = __ballot(mine && ((l >> bit) & 1));
          eq &= ((l >> bit) & 1) ? m : ~m;
        }
        rank[x] = int(__builtin_amdgcn_mbcnt_hi(uint32_t(eq >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(eq), 0u)));
        if (mine) loc[x] = l;
        if (mine && rank[x] == 0) wsc[(x * kChainWaves + wave) * own_cap + l] = uint8_t(__popcll(eq));
      }
    }
    __syncthreads();
    // Exclusive prefix over the slots' counts, kChainThreads slots at a time.
    for (int e0 = 0, run = 0; e0 < nown; e0 += kChainThreads) {
      const int e = e0 + tid;
      int tot = 0;
      if (e < nown)
        for (int w = 0; w < nvw; ++w) tot += wsc[w * own_cap + e];
      int incl = tot;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o);
        if (lane >= o) incl += y;
      }
      if (lane == 63) wtot[wave] = incl;
      __syncthreads();
      int base = run + incl - tot;
#pragma unroll
      for (int w = 0; w < kChainWaves; ++w) {
        base += w < wave ? wtot[w] : 0;
        run += wtot[w];
      }
      if (e < nown) {
        off[e] = uint16_t(base);
        cnt[e] = uint16_t(tot);
      }
      __syncthreads();
    }
#pragma unroll
    for (int x = 0; x < NT; ++x)
      if (x * kChainThreads < n_tok && loc[x] >= 0) {
        int at = off[loc[x]] + rank[x];  // behind the slot's tokens of earlier groups
        for (int w = 0; w < x * kChainWaves + wave; ++w) at += wsc[w * own_cap + loc[x]];
        sorted[at] = uint16_t(x * kChainThreads + tid);
      }
    __syncthreads();
    KVM_TS_A(9);

    // ---- merge + refresh (model/kvm_mixer.py:329-335) of my slots.  A slot
    // that no token was routed to keeps its attention rows: where none of a
    // wave's rows changed (most, once the slots outnumber the tokens) they
    // are copied, keys from LDS and values from the snapshot before.
    const __amdgpu_buffer_rsrc_t skr = l2_rsrc(s_k + srow * D, st.capacity * D * 2);
    const __amdgpu_buffer_rsrc_t svr = l2_rsrc(s_v + srow * D, st.capacity * D * 2);
    const __amdgpu_buffer_rsrc_t slr = l2_rsrc(s_vlen + srow, st.capacity * 4);
    const __amdgpu_buffer_rsrc_t gkr = l2_rsrc(gk_of(i), rowb);
    const __amdgpu_buffer_rsrc_t gvr = l2_rsrc(gv_of(i), rowb);
    const __amdgpu_buffer_rsrc_t ckr = l2_rsrc(cur_k, int64_t(s_after) * D * 2);
    const __amdgpu_buffer_rsrc_t cvr = l2_rsrc(cur_v, int64_t(s_after) * D * 2);
    const __amdgpu_buffer_rsrc_t nk = l2_rsrc(nxt.k + int64_t(row) * nxt.cap * D, int64_t(s_after) * D * 2);
    const __amdgpu_buffer_rsrc_t nv = l2_rsrc(nxt.v + int64_t(row) * nxt.cap * D, int64_t(s_after) * D * 2);
    constexpr int MP = 2;  // slot passes whose loads are in flight together
    for (int l0 = 0; l0 < nown; l0 += MP * RPP) {
      uint4 kk[MP], vv[MP];
      float vl[MP];
      int n[MP], jj[MP];
      bool any[MP];  // uniform: some slot of my wave's rows changed
#pragma unroll
      for (int x = 0; x < MP; ++x) {
        const int l = l0 + x * RPP + sub;
        jj[x] = own_local_to_slot(l, G, member);  // rows at or past s_after lie past the resources
        n[x] = l < nown && jj[x] < s_after ? cnt[l] : 0;
        any[x] = __any(n[x] > 0);
        const int o = (jj[x] * D + part * 8) * 2;
        if (any[x]) {
          kk[x] = l2_ld16(skr, o);
          vv[x] = l2_ld16(svr, o);
          vl[x] = __uint_as_float(l2_ld4(slr, jj[x] * 4));
        } else {
          vv[x] = l2_ld16(cvr, o);
          if (l < OWNL)
            kk[x] = *reinterpret_cast<const uint4 *>(&own_k[l * STR + part * 8]);
          else
            kk[x] = l2_ld16(ckr, o);
        }
      }
#pragma unroll
      for (int x = 0; x < MP; ++x) {
        const int l = l0 + x * RPP + sub;
        if (any[x]) {
          float sk[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
          float sv[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
          const int o = n[x] > 0 ? off[l] : 0;
          for (int i0 = 0; i0 < n[x]; i0 += 4) {
            uint4 xk[4], xv[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              if (i0 + w < n[x]) {
                const int to = (int(sorted[o + i0 + w]) * D + part * 8) * 2;
                xk[w] = l2_ld16(gkr, to);
                xv[w] = l2_ld16(gvr, to);
              }
            }
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              if (i0 + w < n[x]) {
                float fk[8], fv[8];
                unpack8(xk[w], fk);
                unpack8(xv[w], fv);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                  sk[e] += fk[e];
                  sv[e] += fv[e];
                }
              }
            }
          }
          float k[8], v[8];
          unpack8(kk[x], k);
          unpack8(vv[x], v);
          if (n[x] > 0) {  // state = bf16(state + bf16(sum))
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              k[e] = rbf(k[e] + rbf(sk[e]));
              v[e] = rbf(v[e] + rbf(sv[e]));
            }
            const int64_t so = (srow + jj[x]) * D + part * 8;
            store8(s_k + so, k);
            store8(s_v + so, v);
          }
          float ka[8], va[8];
          attn_rows<D>(k, v, vl[x], part, L, ln_w, ln_b, ka, va);
          kk[x] = pack8(ka);
          vv[x] = pack8(va);
          if (l < nown && l < OWNL) *reinterpret_cast<uint4 *>(&own_k[l * STR + part * 8]) = kk[x];
        }
        // Streamed: the attention kernel reads the snapshot much later.
        const uint32_t so = uint32_t((jj[x] * D + part * 8) * 2);
        st16<kPolicyNT>(nk, so, kk[x]);
        st16<kPolicyNT>(nv, so, vv[x]);
      }
    }
    KVM_TS_A(10);
    // My slots' new rows before the next scan: in LDS, and for slots past it
    // in the snapshot.
    if (own_cap > OWNL) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    KVM_TS_A(11);
    KVM_TS_A(12);
  }
}

// ---------------------------------------------------------------------------
// Chain of updates that append nothing (a fixed budget, or a batch in which
// the budget does not grow): routing is split by SLOT instead of by token.
//
// Member m owns the 16-slot blocks m, m + G, m + 2G, ... of its row for the
// whole launch: their sums (s_k, s_v, vlen) and attention key rows live in
// the member's LDS.  Phase p of the launch:
//   prep(p + 1)     merge keys / values of my share of update p + 1's tokens
//                   (while the route keys of update p - 1 are in flight);
//   combine(p - 1)  every member's best slot for every token of update
//                   p - 1 (largest score, then lowest slot);
//   lists(p - 1)    the tokens routed to each of my slots, in token order
//                   (wave ballots: rank within the wave, per-wave counts);
//   merge(p - 1)    sums of the tokens routed to my slots (token order),
//                   refreshed attention rows into LDS and, straight from
//                   registers, into snapshot u0 + p;
//   route(p)        the merge keys of ALL tokens of update p against MY
//                   slots (MFMA 16x16x32 bf16, the per-update kernel's
//                   operand roles and k-step order, so the fp32 scores are
//                   bit-identical) -> per-token maximum over my slots,
//                   published as a tagged partial.
// There is no group barrier per update.  A member publishes its partials
// (score, slot, tag of the update) only after its earlier stores (the
// merge keys / values it prepared) have reached L2 and every wave of the
// workgroup has got there; a reader polls the tags of the partials it
// needs.  Seeing member m's partials of update p therefore also shows that
// m's prepared rows of update p + 1 are readable, and that m has finished
// reading every buffer of update p - 1 (so they may be overwritten).
// Merge keys / values rotate through four buffers (prepared one phase
// ahead, read by route and, a phase later, by the merge); partials
// alternate between two.  Four, not three: a member starts the prep of
// update p + 1 (into buffer (p + 1) % 4) before it has seen the partials of
// update p - 1, so another member may still be in phase p - 1, gathering
// the rows of update p - 2 and loading route operands of update p - 1,
// while a member already in phase p + 1 may be preparing update p + 2; with
// three buffers update p + 1 would share the buffer of update p - 2.  The
// two partial buffers suffice: a member publishes update p only after it
// has seen every member's partials of update p - 1, by which time every
// member has stopped polling those of update p - 2.  The raw tokens a prep needs are loaded at the
// end of the phase before; the route operands of update p are loaded once
// the merge's gathered rows have arrived, so they never queue in L2 ahead
// of the gathers.
constexpr int kOwnMax = 128;      // owned slots per member at most (8 blocks of 16)
constexpr int kTokWave = 64;      // tokens per wave in route(p)
constexpr int kFixedMaxTok = kChainWaves * kTokWave;  // == kChainThreads: one token per thread


// GM: the group size G (8 or 16); OWN: owned slots per member the LDS holds
// (64, or 128 for states of up to 1024 slots at G = 8).
template <int D, int GM, int OWN>
__global__ __launch_bounds__(kChainThreads) void k_chain_fixed(
    kvm_layer L, kvm_seq src, int n_tok, kvm_state st, SnapRing snaps, ChainList list,
    ChainScratch cs, int rows, int row0, int nrows, int32_t *route_log, int32_t *append_log,
    int64_t log_stride) {
  constexpr int GL = D / 8;                 // lanes per D-wide row
  constexpr int STR = D + 8;                // LDS row stride of key rows (elements)
  constexpr int KS = D / 32;
  constexpr int RPP = kChainThreads / GL;   // rows per pass
  constexpr int SP = OWN / RPP;             // passes over the owned slots
  constexpr int HP = SP < 2 ? SP : 2;       // passes per half (the sums of one half live in registers)
  constexpr int NH = SP / HP;               // halves of the owned slots
  // Routed token rows staged in LDS at once (96 at OWN 128 and D 128, where
  // the owned rows need the room).
  constexpr int STAGE = (OWN == 128 && D == 128) ? 96 : 128;
  constexpr int RPI = 1024 / (2 * D);        // token rows per 1 KiB DMA instruction
  constexpr int KI = STAGE / RPI;            // DMA instructions per staged chunk (keys or values)
  constexpr int LOG2_OWN = OWN == 128 ? 7 : 6;
  static_assert(OWN == 64 || OWN == 128, "owned slots");
  static_assert(SP == NH * HP, "refresh halves");
  static_assert(kChainTok <= STAGE, "raw rows alias the staging buffers");
  constexpr int IT = RawTok<D>::IT;         // passes over the member's prep tokens
  constexpr int NRAW = 2 * (kChainTok / RPI) / kChainWaves;  // raw-row DMA instructions per wave
  static_assert(NRAW * kChainWaves == 2 * (kChainTok / RPI), "raw DMA split");
  __shared__ __attribute__((aligned(16))) uint16_t own_k[OWN * STR];  // attention keys
  __shared__ __attribute__((aligned(16))) uint16_t own_sk[OWN * D];   // key sums
  __shared__ __attribute__((aligned(16))) uint16_t own_sv[OWN * D];   // value sums
  // Routed token rows of the merge.  The raw key / value rows of my prep
  // share of an update share these buffers: they are DMA'd during a phase's
  // route, after that phase's sums have read the staged rows, and read by
  // the next phase's prep, before that phase's gathers are issued.
  __shared__ __attribute__((aligned(16))) uint16_t stage_k[STAGE * D];
  __shared__ __attribute__((aligned(16))) uint16_t stage_v[STAGE * D];
  uint16_t *const raw_k = stage_k;
  uint16_t *const raw_v = stage_v;
  __shared__ float own_vl[OWN];
  __shared__ int tok_lds[kChainMax];  // first token of each update (list.tok_begin)
  __shared__ int sorted[kFixedMaxTok];
  __shared__ int wsc[kChainWaves][OWN];  // per-wave slot counts
  __shared__ int cnt[OWN], off[OWN];
  __shared__ int ok_lds;
  __shared__ float ln_w[D], ln_b[D];  // ln_s_k parameters (LDS: no wait on global loads)

  constexpr int G = GM;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, part = tid % GL;
  const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
  const int member = q % G, group = (q / G) * 8 + xcd;
  if (group >= nrows) return;
  const int row = row0 + group;  // this launch serves rows row0 .. row0 + nrows - 1
  const int b = row / int(L.kv_heads), h = row % int(L.kv_heads);
  const int64_t rb = int64_t(row) * n_tok;
  // Per-row bases; the buffers of one kind lie a 32-bit stride apart (the host
  // launches the chain only when they fit).
  const int buf_stride = rows * n_tok * D;   // elements between merge buffers
  const int part_stride = rows * n_tok * G;  // partials between the two buffers
  uint16_t *const gk_row = cs.gk + rb * D;
  uint16_t *const gv_row = cs.gv + rb * D;
  uint2 *const part_row = cs.part + rb * G;
  uint16_t *const snk_row = snaps.k + int64_t(row) * snaps.cap * D;
  uint16_t *const snv_row = snaps.v + int64_t(row) * snaps.cap * D;
  const int snap_stride = int(snaps.stride);
  const int snap_bytes = int(snaps.cap) * D * 2;
  const int k_st = int(src.k_st), v_st = int(src.v_st), g_st = int(src.g_st);
  const int tpm = (n_tok + G - 1) / G;                   // prep tokens per member (<= 64)
  const int pt0 = member * tpm;
  const int pnt = max(0, min(n_tok, pt0 + tpm) - pt0);
  unsigned *ctr = cs.bar + group * kCounterStride;
  unsigned target = 0;
  auto arrive = [&]() __attribute__((always_inline)) {
    target += unsigned(G);
    group_arrive(ctr);
  };
  auto wait = [&]() __attribute__((always_inline)) {
    return group_wait(ctr, target, cs, &ok_lds);
  };
  uint16_t *s_k = static_cast<uint16_t *>(st.s_k);
  uint16_t *s_v = static_cast<uint16_t *>(st.s_v);
  float *s_vlen = static_cast<float *>(st.s_vlen);
  const int64_t srow = int64_t(row) * st.capacity;
  const int S = list.state_before[0];  // no appends: constant over the batch
  const int protect = min(int(L.sink_len), S);
  // Owned local slots: 16 per owned block below S.
  const int nblk = (S + 15) >> 4;
  const int nown = member < nblk ? ((nblk - 1 - member) / G + 1) * 16 : 0;
  const uint16_t *k_row = static_cast<const uint16_t *>(src.k) + b * src.k_sb + h * src.k_sh;
  const uint16_t *v_row = static_cast<const uint16_t *>(src.v) + b * src.v_sb + h * src.v_sh;
  const uint16_t *g_row = static_cast<const uint16_t *>(src.gate) + b * src.g_sb + h * src.g_sh;

  for (int d = tid; d < D; d += kChainThreads) {
    ln_w[d] = static_cast<const float *>(L.ln_weight)[d];
    ln_b[d] = static_cast<const float *>(L.ln_bias)[d];
  }
  // The first token of every update, read from LDS where the raw rows are
  // fetched (a scalar load of the kernel argument would wait for memory).
  for (int i = tid; i < list.count; i += kChainThreads) tok_lds[i] = list.tok_begin[i];
  // ---- owned state and attention keys into LDS (slots >= S stay zero).
  {
    const AttnRows a0 = snap_at(snaps, list.u0);
    for (int base = 0; base < OWN; base += RPP) {
      const int l = base + tid / GL;
      const int j = own_local_to_slot(l, G, member);
      const bool valid = l < nown && j < S;
      const uint4 z = make_uint4(0, 0, 0, 0);
      const int64_t so = (srow + j) * D + part * 8;
      *reinterpret_cast<uint4 *>(&own_sk[l * D + part * 8]) =
          valid ? *reinterpret_cast<const uint4 *>(s_k + so) : z;
      *reinterpret_cast<uint4 *>(&own_sv[l * D + part * 8]) =
          valid ? *reinterpret_cast<const uint4 *>(s_v + so) : z;
      *reinterpret_cast<uint4 *>(&own_k[l * STR + part * 8]) =
          valid ? *reinterpret_cast<const uint4 *>(a0.k + (int64_t(row) * a0.cap + j) * D + part * 8)
                : z;
      if (part == 0) own_vl[l] = valid ? s_vlen[srow + j] : 0.f;
    }
  }

  // Raw key / value rows of my prep share of update i go from device memory
  // straight into LDS (non-temporal DMA, no registers): wave w issues
  // instructions w, w + 8, ... of the keys, then of the values, each filling
  // RPI consecutive rows; rows past my share lie past the resource and read
  // zero.  The gates go into registers.  Issued a whole phase before the prep
  // that reads them, so the prep never waits for device memory.  Prefill
  // tokens never come from a ring (src.ring == 0, checked by the host).
  uint16_t rg[IT];
  auto raw_dma = [&](int i) __attribute__((always_inline)) {
    const int64_t tb = int64_t(__builtin_amdgcn_readfirstlane(tok_lds[i])) + pt0;
    const int kb = pnt > 0 ? ((pnt - 1) * k_st + D) * 2 : 0;
    const int vb = pnt > 0 ? ((pnt - 1) * v_st + D) * 2 : 0;
    const __amdgpu_buffer_rsrc_t kr = l2_rsrc(k_row + tb * k_st, kb);
    const __amdgpu_buffer_rsrc_t vr = l2_rsrc(v_row + tb * v_st, vb);
    const uint32_t kbase = lds_addr(raw_k), vbase = lds_addr(raw_v);
#pragma unroll
    for (int t = 0; t < NRAW; ++t) {
      const int c = __builtin_amdgcn_readfirstlane(wave) + kChainWaves * t;
      constexpr int KIR = kChainTok / RPI;
      const int ci = c < KIR ? c : c - KIR;
      const int r = ci * RPI + lane / GL;
      if (c < KIR)
        dma16_nt(kr, kbase + uint32_t(ci * 1024), uint32_t((r * k_st + part * 8) * 2));
      else
        dma16_nt(vr, vbase + uint32_t(ci * 1024), uint32_t((r * v_st + part * 8) * 2));
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int lt = (tid + it * kChainThreads) / GL;
      rg[it] = g_row[tb * g_st + (lt < pnt ? lt : 0) * g_st];
    }
  };
  // prep (model/kvm_mixer.py:120-129, model/kvm_triton_mixer.py:429-446):
  // merge key / value rows of my share of update i (from the raw rows in
  // LDS), packed bf16, stored into merge buffer i % 4.
  auto prep = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int lt = (tid + it * kChainThreads) / GL;
      float k[8], v[8];
      unpack8(*reinterpret_cast<const uint4 *>(&raw_k[lt * D + part * 8]), k);
      unpack8(*reinterpret_cast<const uint4 *>(&raw_v[lt * D + part * 8]), v);
      const float g = bf2f(rg[it]);
      prep_key<D>(k, part, L, ln_w, ln_b);
      float gk[8], gv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        gk[e] = L.gate_keys ? k[e] * g : k[e];
        gv[e] = L.gate_values ? v[e] * g : v[e];
      }
      if (lt < pnt) {
        const uint32_t o = uint32_t(((pt0 + lt) * D + part * 8) * 2);
        st16<0>(l2_rsrc(gk_row + (i % 4) * buf_stride, n_tok * D * 2), o, pack8(gk));
        st16<0>(l2_rsrc(gv_row + (i % 4) * buf_stride, n_tok * D * 2), o, pack8(gv));
      }
    }
  };
  // Tag of the partials of update i (never 0: the entries are cleared to 0
  // at the start of a launch, so a workspace's old contents never match).
  auto tag_of = [](int i) __attribute__((always_inline)) { return uint32_t(0x8000u | uint32_t(i)); };
  __shared__ int fail_lds;

  // Prologue: prep(0), then the raw rows of update 1; the group barrier's
  // store wait (vmcnt(0)) also completes that DMA, and its workgroup barrier
  // makes the rows visible to every wave.
  __syncthreads();  // tok_lds, ln_w / ln_b and the owned rows are in LDS
  raw_dma(0);
  if (tid == 0) fail_lds = 0;
  // My partials in both buffers start cleared.
  for (int t = tid; t < n_tok; t += kChainThreads) {
    cs.part[rb * G + int64_t(t) * G + member] = make_uint2(0u, 0u);
    cs.part[part_stride + rb * G + int64_t(t) * G + member] = make_uint2(0u, 0u);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  prep(0);
  __syncthreads();  // every wave has read the raw rows of update 0
  if (list.count > 1) raw_dma(1);
  arrive();
  if (!wait()) return;

  int snap_i = int(int64_t(list.u0) % snaps.ring);  // ring entry of snapshot u0 + p
  for (int p = 0; p <= list.count; ++p) {
    KVM_TS(0);
    const bool do_route = p < list.count;
    const bool do_prep = p + 1 < list.count;
    // Route operands of update p: my wave's 64 tokens (tokens >= n_tok read zero).
    uint4 bx[4][KS];
    auto load_bx = [&](int tt0, int tt1, int ks0, int ks1) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t gr =
          l2_rsrc(gk_row + (p % 4) * buf_stride, n_tok * D * 2);
#pragma unroll
      for (int tt = tt0; tt < tt1; ++tt)
#pragma unroll
        for (int ks = ks0; ks < ks1; ++ks)
          bx[tt][ks] = l2_ld16(gr, ((wave * kTokWave + tt * 16 + (lane & 15)) * D + ks * 32 +
                                    (lane >> 4) * 8) * 2);
    };
    // Partials of update p - 1 for my token (tokens >= n_tok read zero and
    // are not waited for).
    uint4 pw[GM / 2];
    const __amdgpu_buffer_rsrc_t pr =
        l2_rsrc(part_row + ((p - 1) & 1) * part_stride, n_tok * G * 8);
    if (p >= 1) {
#pragma unroll
      for (int i = 0; i < GM / 2; ++i) pw[i] = l2_ld16(pr, (tid * GM + 2 * i) * 8);
    }
    // The next update's prep (raw rows already in LDS) while that load is
    // in flight.
    if (do_prep) prep(p + 1);
    if (p == 0) {
      load_bx(0, 4, 0, KS);
      __syncthreads();  // every wave has read the raw rows of update 1
    }
    KVM_TS(1);

    if (p >= 1) {
      // ---- combine(p - 1) and the lists of my slots.
      const int pi = p - 1;
      const int64_t u = int64_t(list.u0) + pi;
      // Wait (bounded) until every member's partial of my token carries the
      // tag of update p - 1, then keep the first argmax: larger score, then
      // lower slot (scores are MFMA sums started at +0, never -0 or NaN).
      bool ok_tok = false;
      {
        const uint32_t want = tag_of(pi);
        bool ok = tid >= n_tok;
        unsigned polls = 0;
        for (;;) {
          bool fresh = true;
#pragma unroll
          for (int i = 0; i < GM / 2; ++i) fresh &= (pw[i].y >> 16) == want && (pw[i].w >> 16) == want;
          ok |= fresh;
          if (__all(ok) || polls >= cs.max_polls) break;
          if ((polls & 255u) == 255u &&
              __hip_atomic_load(cs.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            break;
          __builtin_amdgcn_s_sleep(1);
          ++polls;
          if (!ok) {
#pragma unroll
            for (int i = 0; i < GM / 2; ++i) pw[i] = l2_ld16(pr, (tid * GM + 2 * i) * 8);
          }
        }
        ok_tok = ok && tid < n_tok;
        KVM_TS(7);
        if (!__all(ok)) {
          if ((tid & 63) == 0) {
            __hip_atomic_store(cs.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_or(cs.status, unsigned(KVM_STATUS_CHAIN_TIMEOUT), __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
            fail_lds = 1;
          }
        }
      }
      // The route operands of update p: every member stores its prepared
      // rows of update p before it publishes any partial of update p - 1,
      // so they are in L2 now.  Issued here, while the memory pipeline is
      // otherwise idle during the lists, they have landed long before the
      // gathers behind them are waited for.
      // The first half of the k-steps here, the rest in two quarters at the
      // refresh passes: a CU's vector memory pipeline moves about 64 bytes
      // per clock, so a burst of all of them would stall the issuing waves
      // and delay the gathers queued behind them.
      if (do_route) load_bx(0, 4, 0, KS / 2);
      KVM_TS(14);
      // Partials are route keys (see route(p)): the largest wins.
      uint64_t best = 0;
#pragma unroll
      for (int i = 0; i < GM / 2; ++i) {
        const uint64_t k0 = (uint64_t(pw[i].x) << 32) | (pw[i].y & 0xffffu);
        const uint64_t k1 = (uint64_t(pw[i].z) << 32) | (pw[i].w & 0xffffu);
        best = k0 > best ? k0 : best;
        best = k1 > best ? k1 : best;
      }
      int bi = (best >> 32) != 0 ? int(0xffffu - uint32_t(best & 0xffffu)) : -1;
      if (!ok_tok) bi = -1;  // past n_tok, or a partial that never arrived
      const bool mine = bi >= 0 && ((bi >> 4) % G) == member;
      const int my_loc = mine ? ((((bi >> 4) / G) << 4) | (bi & 15)) : -1;
      if (tid >= pt0 && tid < pt0 + pnt) {  // each member logs its prep share
        if (route_log) route_log[u * log_stride + rb + tid] = bi;
        if (append_log) append_log[u * log_stride + rb + tid] = 0;
      }
      // Tokens of my wave with the same local slot (ballots over its bits):
      // rank among them, and their count from the group's first lane.  A
      // wave's LDS stores complete in order, so the clear of its own row of
      // wsc precedes the counts it writes.
#pragma unroll
      for (int c = 0; c < OWN; c += 64) wsc[wave][c + lane] = 0;
      uint64_t eq = __ballot(mine);
#pragma unroll
      for (int bit = 0; bit < LOG2_OWN; ++bit) {
        const uint64_t m = __ballot(mine && ((my_loc >> bit) & 1));
        eq &= ((my_loc >> bit) & 1) ? m : ~m;
      }
      const int rank = int(__builtin_amdgcn_mbcnt_hi(uint32_t(eq >> 32),
                                                     __builtin_amdgcn_mbcnt_lo(uint32_t(eq), 0u)));
      if (mine && rank == 0) wsc[wave][my_loc] = __popcll(eq);
      __syncthreads();
      if (fail_lds) return;  // a partial never arrived: the launch is abandoned
      KVM_TS(15);
      // Every wave computes the exclusive prefix over slots (slot e's first
      // list position, and its position after the tokens of lower waves)
      // itself, so that each places its own tokens without another barrier;
      // wave 0 also keeps off / cnt for the sums.
      int ntot;  // tokens routed to my slots
      {
        constexpr int PER = OWN / 64;  // consecutive slots per lane
        int run[PER], mine_pre[PER], tot = 0;
#pragma unroll
        for (int x = 0; x < PER; ++x) {
          const int e = lane * PER + x;
          run[x] = 0;
          mine_pre[x] = 0;
#pragma unroll
          for (int w = 0; w < kChainWaves; ++w) {
            if (w == wave) mine_pre[x] = run[x];
            run[x] += wsc[w][e];
          }
          tot += run[x];
        }
        int incl = tot;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int y = __shfl_up(incl, o);
          if (lane >= o) incl += y;
        }
        int base = incl - tot;
        int pos[PER];
#pragma unroll
        for (int x = 0; x < PER; ++x) {
          if (wave == 0) {
            off[lane * PER + x] = base;
            cnt[lane * PER + x] = run[x];
          }
          pos[x] = base + mine_pre[x];
          base += run[x];
        }
        ntot = __shfl(incl, 63);
        int at = 0;
#pragma unroll
        for (int x = 0; x < PER; ++x) {
          const int v = __shfl(pos[x], (mine ? my_loc : 0) / PER);
          if ((mine ? my_loc : 0) % PER == x) at = v;
        }
        if (mine) sorted[at + rank] = tid;
      }
      __syncthreads();
      KVM_TS(2);

      // ---- merge(p - 1) (model/kvm_mixer.py:329-335).  The routed token
      // rows are staged in LDS (all loads of a chunk in flight together),
      // then each slot sums its rows in token order.
      const __amdgpu_buffer_rsrc_t gkr =
          l2_rsrc(gk_row + (pi % 4) * buf_stride, n_tok * D * 2);
      const __amdgpu_buffer_rsrc_t gvr =
          l2_rsrc(gv_row + (pi % 4) * buf_stride, n_tok * D * 2);
      // Sums of the half of my slots being merged (registers for HP passes).
      float sk[HP][8], sv[HP][8];
      // Routed rows are staged STAGE at a time, straight from L2 into LDS
      // (device-scope LDS-DMA loads, no registers).  Wave w fills staged rows
      // RPI*ci .. RPI*ci + RPI - 1 for ci = w, w + 8, ...: the token indices
      // of all its instructions are read from LDS first (one wait), then the
      // key and the value row of each are issued.  Rows past ntot point past
      // the resource and are not written.
      auto gather = [&](int c0) __attribute__((always_inline)) {
        const uint32_t kbase = lds_addr(stage_k), vbase = lds_addr(stage_v);
        const int w0 = __builtin_amdgcn_readfirstlane(wave);
        constexpr int NG = KI / kChainWaves;
        static_assert(NG * kChainWaves == KI, "gather split");
        uint32_t to[NG];
#pragma unroll
        for (int t = 0; t < NG; ++t) {
          const int pos = c0 + (w0 + kChainWaves * t) * RPI + lane / GL;
          const int tok = sorted[min(pos, kFixedMaxTok - 1)];
          // Rows past ntot point past the resource (n_tok) and are not written.
          to[t] = uint32_t(((pos < ntot ? tok : n_tok) * D + part * 8) * 2);
        }
#pragma unroll
        for (int t = 0; t < NG; ++t) {
          const int ci = w0 + kChainWaves * t;
          if (c0 + ci * RPI < ntot) {  // instructions wholly past ntot are not issued
            dma16_l2(gkr, kbase + uint32_t(ci * 1024), to[t]);
            dma16_l2(gvr, vbase + uint32_t(ci * 1024), to[t]);
          }
        }
      };
      // Adds the staged rows c0 .. of the slots of half h to the sums, in
      // token order; `arrived`: wait for this wave's gathers, then for every
      // wave's (not needed when the rows were staged for an earlier half);
      // `release`: a barrier after the reads, before another gather reuses
      // the staging buffers (the merge's final barrier covers the last use).
      auto stage_sum = [&](int c0, int h, bool arrived, bool release) __attribute__((always_inline)) {
        const int nrow = min(STAGE, ntot - c0);
        if (arrived) {
          wait_vm<0>();
          __syncthreads();
        }
#pragma unroll
        for (int sp = 0; sp < HP; ++sp) {
          const int l = (h * HP + sp) * RPP + tid / GL;
          if (l < nown) {
            const int e0 = max(off[l], c0), e1 = min(off[l] + cnt[l], c0 + nrow);
            auto add_row = [&](uint4 rk, uint4 rv) __attribute__((always_inline)) {
              float fk[8], fv[8];
              unpack8(rk, fk);
              unpack8(rv, fv);
#pragma unroll
              for (int x = 0; x < 8; ++x) {
                sk[sp][x] += fk[x];
                sv[sp][x] += fv[x];
              }
            };
            auto row_k = [&](int e) { return *reinterpret_cast<const uint4 *>(&stage_k[(e - c0) * D + part * 8]); };
            auto row_v = [&](int e) { return *reinterpret_cast<const uint4 *>(&stage_v[(e - c0) * D + part * 8]); };
            int e = e0;
            if constexpr (OWN == 128) {
              // Four rows' LDS reads in flight at once: at 1024 slots the
              // routes are uneven enough that some slots sum tens of rows.
              // Still added in token order.
              for (; e + 4 <= e1; e += 4) {
                uint4 rk[4], rv[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                  rk[u] = row_k(e + u);
                  rv[u] = row_v(e + u);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) add_row(rk[u], rv[u]);
              }
            }
            for (; e < e1; ++e) add_row(row_k(e), row_v(e));
          }
        }
        if (release) __syncthreads();
      };
      // Refreshed attention rows: keys into LDS (route operands), keys and
      // values into snapshot u0 + p straight from registers (non-temporal:
      // the attention kernel reads them much later), and after the batch's
      // last update also into the state's attention rows.
      // Snapshot u0 + p: ring entry snap_i (advanced by one per phase).
      const __amdgpu_buffer_rsrc_t nk =
          l2_rsrc(snk_row + int64_t(snap_i) * snap_stride, snap_bytes);
      const __amdgpu_buffer_rsrc_t nv =
          l2_rsrc(snv_row + int64_t(snap_i) * snap_stride, snap_bytes);
      const bool fin = !do_route && list.final_rows != 0;
      uint16_t *s_ka = static_cast<uint16_t *>(st.s_k_attn);
      uint16_t *s_va = static_cast<uint16_t *>(st.s_v_attn);
      auto refresh = [&](int h) __attribute__((always_inline)) {
#pragma unroll
        for (int sp = 0; sp < HP; ++sp) {
          const int l = (h * HP + sp) * RPP + tid / GL;
          const int j = own_local_to_slot(l, G, member);
          const bool valid = l < nown && j < S;
          float k[8], v[8];
          unpack8(*reinterpret_cast<const uint4 *>(&own_sk[l * D + part * 8]), k);
          unpack8(*reinterpret_cast<const uint4 *>(&own_sv[l * D + part * 8]), v);
          if (valid && cnt[l] > 0) {  // state = bf16(state + bf16(sum))
            round_pack8(sk[sp]);
            round_pack8(sv[sp]);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              k[e] += sk[sp][e];
              v[e] += sv[sp][e];
            }
            *reinterpret_cast<uint4 *>(&own_sk[l * D + part * 8]) = round_pack8(k);
            *reinterpret_cast<uint4 *>(&own_sv[l * D + part * 8]) = round_pack8(v);
          }
          // Attention rows of the slot (kvm_seq.hpp attn_rows, in two steps;
          // the rows are only stored, so they are rounded by the packing).
          float ka[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) ka[e] = k[e];
          layer_norm8<D>(ka, part, ln_w, ln_b, float(L.ln_eps));
          const uint4 kk = pack8(ka);
          const uint4 vv = attn_value8_packed<D>(v, own_vl[l]);
          if (valid) {
            *reinterpret_cast<uint4 *>(&own_k[l * STR + part * 8]) = kk;
            const uint32_t ao = uint32_t((j * D + part * 8) * 2);
            st16<kPolicyNT>(nk, ao, kk);
            st16<kPolicyNT>(nv, ao, vv);
            if (fin) {
              const int64_t so = (srow + j) * D + part * 8;
              *reinterpret_cast<uint4 *>(s_ka + so) = kk;
              *reinterpret_cast<uint4 *>(s_va + so) = vv;
            }
          }
          __builtin_amdgcn_sched_barrier(0);  // one slot pass at a time (register pressure)
          if (h == NH - 1 && sp == 0) {
            KVM_TS(11);
            if (do_route) load_bx(0, 4, KS * 3 / 4, KS);  // the last quarter of the route operands
          }
        }
      };
      auto zero_sums = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int sp = 0; sp < HP; ++sp)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            sk[sp][e] = 0.f;
            sv[sp][e] = 0.f;
          }
      };
      gather(0);
      KVM_TS(8);
      if (ntot <= STAGE) {  // one staged round serves every half
#pragma unroll 1
        for (int h = 0; h < NH; ++h) {
          zero_sums();
          stage_sum(0, h, h == 0, false);
          if (h == 0) {
            KVM_TS(9);
            KVM_TS(10);
          }
          // The third quarter of the route operands with the last half (not
          // earlier: with them resident the earlier halves' sums would spill).
          if (h == NH - 1 && do_route) load_bx(0, 4, KS / 2, KS * 3 / 4);
          refresh(h);
        }
      } else {  // several rounds: each half gathers them again
#pragma unroll 1
        for (int h = 0; h < NH; ++h) {
          zero_sums();
          for (int c0 = 0; c0 < ntot; c0 += STAGE) {
            if (h > 0 || c0 > 0) gather(c0);
            stage_sum(c0, h, true, true);
          }
          if (h == NH - 1 && do_route) load_bx(0, 4, KS / 2, KS * 3 / 4);
          refresh(h);
          __syncthreads();  // every wave has read the staged rows before the next gather
        }
      }
      __syncthreads();
    }
    KVM_TS(3);

    if (do_route) {
      // ---- route(p) (model/kvm_fp32_routing_reference.py:30-34) against my
      // slots: per-lane maximum in increasing slot order (strict >), then
      // across the lane groups; larger score wins, ties go to the lower slot.
      float best[4];
      int bidx[4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        best[tt] = -INFINITY;
        bidx[tt] = -1;
      }
      for (int lt = 0; lt < nown; lt += 16) {
        const int jb = own_local_to_slot(lt, G, member);  // first slot of the block
        uint4 a[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          a[ks] = *reinterpret_cast<const uint4 *>(
              &own_k[(lt + (lane & 15)) * STR + ks * 32 + (lane >> 4) * 8]);
        const bool scan = needs_scan(a[0], jb, protect, S);
        // k-steps outermost: the four token tiles' accumulations interleave
        // (each still sums its k-steps in order).
        f32x4 accs[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) accs[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int tt = 0; tt < 4; ++tt)
            accs[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[ks]), as_bf16x8(bx[tt][ks]),
                                                               accs[tt], 0, 0, 0);
        // The raw rows of update p + 2 once the first block's products have
        // been issued: every route operand has arrived by then, so the DMA
        // queues behind nothing the route waits for, and the release wait
        // below completes it (every wave read the raw rows of update p + 1
        // at the start of this phase, before the lists' barriers).
        if (lt == 0 && p + 2 < list.count) {
          __builtin_amdgcn_sched_barrier(0);
          raw_dma(p + 2);
          __builtin_amdgcn_sched_barrier(0);
        }
        const int j0 = jb + (lane >> 4) * 4;  // slot of acc[0]
        if (scan) {
#pragma unroll
          for (int tt = 0; tt < 4; ++tt) scan_max4(accs[tt], j0, protect, S, best[tt], bidx[tt]);
        } else {
#pragma unroll
          for (int tt = 0; tt < 4; ++tt) keep_max4(accs[tt], j0, best[tt], bidx[tt]);
        }
      }
      KVM_TS(12);
      if (nown == 0 && p + 2 < list.count) raw_dma(p + 2);  // a member without slots
      // Release: this member's earlier stores (its prepared rows of update
      // p + 1) are in L2 before any of its partials of update p is.
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      KVM_TS(13);
      // Partials are route keys: {mono(score), tag << 16 | (0xffff - slot)},
      // compared as 64-bit integers (the tags are equal), so the maximum is
      // the largest score and, among equal scores, the lowest slot; no
      // candidate is {0, tag << 16}, below every real key.
      const uint32_t tg = tag_of(p) << 16;
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const uint32_t bu = __float_as_uint(best[tt]);
        uint32_t khi = bidx[tt] >= 0 ? ((bu & 0x80000000u) ? ~bu : (bu | 0x80000000u)) : 0u;
        uint32_t klo = bidx[tt] >= 0 ? 0xffffu - uint32_t(bidx[tt]) : 0u;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const uint32_t ohi = r == 0 ? xor16_lane(khi, lane) : xor32_lane(khi, lane);
          const uint32_t olo = r == 0 ? xor16_lane(klo, lane) : xor32_lane(klo, lane);
          const uint64_t mine = (uint64_t(khi) << 32) | klo, other = (uint64_t(ohi) << 32) | olo;
          const bool take = other > mine;
          khi = take ? ohi : khi;
          klo = take ? olo : klo;
        }
        const int t = wave * kTokWave + tt * 16 + lane;
        if (lane < 16 && t < n_tok)
          __builtin_amdgcn_raw_buffer_store_b64(
              __builtin_bit_cast(__attribute__((ext_vector_type(2))) unsigned, make_uint2(khi, tg | klo)),
              l2_rsrc(part_row + (p & 1) * part_stride, n_tok * G * 8), (t * G + member) * 8, 0, 0);
      }
      KVM_TS(4);
      KVM_TS(5);
      KVM_TS(6);
    }
    snap_i = snap_i + 1 == int(snaps.ring) ? 0 : snap_i + 1;
  }

  // ---- owned state back to the caller's arrays.
  for (int base = 0; base < nown; base += RPP) {
    const int l = base + tid / GL;
    if (l < nown) {
      const int j = own_local_to_slot(l, G, member);
      if (j < S) {
        const int64_t so = (srow + j) * D + part * 8;
        *reinterpret_cast<uint4 *>(s_k + so) = *reinterpret_cast<const uint4 *>(&own_sk[l * D + part * 8]);
        *reinterpret_cast<uint4 *>(s_v + so) = *reinterpret_cast<const uint4 *>(&own_sv[l * D + part * 8]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The chain without appends when there are rows for every compute unit: one
// workgroup per row, no exchange.  The slot-owner kernel above spends most of
// an update on the latency of its exchange (7.8 us at 32 slots and 32 tokens
// per member, C 256, 256 slots), and runs 8 launches of 32 rows for 256 rows;
// here a row's work is done in one place and every launch is full: less than
// half the time at 256 rows (figures at fixed_group).  Bound by VALU issue
// (the LayerNorms and sums of C tokens and S slots; VALU busy 80 % of the
// compute units' busy cycles): of 32 us, prep 4.2, route 8.8 (its key
// fragments from LDS at 64 B per clock as much), lists 3.2, keys 7.4, values
// 1.7 + 6.9.
// 16 waves of 128 registers: with 8 waves of 256 the phases but the route
// were slower (34.8 us).
//
// LDS holds the attention keys of every slot and one update's token rows
// (merge keys, then, once every slot has summed its keys, merge values in the
// same place); the sums s_k / s_v live in registers for the whole launch,
// packed bf16, a slot's row in the D/8 lanes that refresh it.  One update:
//   prep     merge keys of the C tokens (raw rows loaded during the update
//            before) into LDS; the raw values are fetched behind it
//   route    MFMA, waves = token groups of 32 x slot groups; a token's best
//            (score, slot) of each slot group through LDS
//   lists    the tokens of each slot in token order (ballots, prefix sums)
//   keys     fp32 sums in token order, LayerNorm, own_k and snapshot rows
//   values   gated value rows into LDS, sums, value rows of the snapshot
// The same arithmetic, in the same order, as the kernels above.
constexpr int kRowThreads = 1024;
constexpr int kRowWaves = kRowThreads / 64;
constexpr int kRowPasses = 4;  // slot (and token) rows per thread
constexpr int kRowTiles = 2;   // 16-token tiles per wave in the route

template <int D>
struct RowMax {  // slots, and tokens per update, that LDS and the registers hold
  static constexpr int value = kRowPasses * (kRowThreads / (D / 8));
};

template <int D>
__global__ __launch_bounds__(kRowThreads) void k_chain_row(
    kvm_layer L, kvm_seq src, int n_tok, kvm_state st, SnapRing snaps, ChainList list, int32_t *route_log,
    int32_t *append_log, int64_t log_stride) {
  constexpr int GL = D / 8;
  constexpr int STR = D + 8;
  constexpr int KS = D / 32;
  constexpr int RPP = kRowThreads / GL;  // rows per pass
  constexpr int NP = kRowPasses;
  constexpr int MAX = RowMax<D>::value;
  __shared__ __attribute__((aligned(16))) uint16_t own_k[MAX * STR];  // attention keys
  __shared__ __attribute__((aligned(16))) uint16_t tok[MAX * STR];    // merge keys, then merge values
  constexpr int TT = kRowTiles;
  constexpr int LW = MAX / 64;  // waves whose threads have a token in the lists
  // Route keys [slot group][token] (kRowWaves * 16 TT of them), then each wave's slot counts.
  __shared__ __attribute__((aligned(16)))
  uint64_t scratch[kRowWaves * 16 * TT > LW * MAX / 4 ? kRowWaves * 16 * TT : LW * MAX / 4];
  __shared__ uint16_t sorted[MAX], off[MAX], cnt[MAX];
  __shared__ int wtot[kRowWaves];
  __shared__ int tok_lds[kChainMax];
  __shared__ float own_vl[MAX];
  __shared__ float ln_w[D], ln_b[D];
  uint16_t *const wsc = reinterpret_cast<uint16_t *>(scratch);  // [LW][MAX]

  const int tid = threadIdx.x, lane = tid & 63, part = tid % GL, sub = tid / GL;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = blockIdx.x;
  const int b = row / int(L.kv_heads), h = row % int(L.kv_heads);
  const int S = list.state_before[0];  // no appends: constant over the batch
  const int protect = min(int(L.sink_len), S);
  const int nblk = (S + 15) >> 4;
  const int64_t srow = int64_t(row) * st.capacity;
  const uint16_t *k_row = static_cast<const uint16_t *>(src.k) + b * src.k_sb + h * src.k_sh;
  const uint16_t *v_row = static_cast<const uint16_t *>(src.v) + b * src.v_sb + h * src.v_sh;
  const uint16_t *g_row = static_cast<const uint16_t *>(src.gate) + b * src.g_sb + h * src.g_sh;
  uint16_t *s_k = static_cast<uint16_t *>(st.s_k), *s_v = static_cast<uint16_t *>(st.s_v);
  uint16_t *s_ka = static_cast<uint16_t *>(st.s_k_attn), *s_va = static_cast<uint16_t *>(st.s_v_attn);

  for (int d = tid; d < D; d += kRowThreads) {
    ln_w[d] = static_cast<const float *>(L.ln_weight)[d];
    ln_b[d] = static_cast<const float *>(L.ln_bias)[d];
  }
  for (int i = tid; i < list.count; i += kRowThreads) tok_lds[i] = list.tok_begin[i];
  // Sums of slot p * RPP + sub in registers; attention keys and vlen in LDS.
  uint4 sk[NP], sv[NP];
  {
    const AttnRows a0 = snap_at(snaps, list.u0);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int j = p * RPP + sub;
      sk[p] = sv[p] = make_uint4(0, 0, 0, 0);
      if (j < S) {
        sk[p] = *reinterpret_cast<const uint4 *>(s_k + (srow + j) * D + part * 8);
        sv[p] = *reinterpret_cast<const uint4 *>(s_v + (srow + j) * D + part * 8);
        *reinterpret_cast<uint4 *>(&own_k[j * STR + part * 8]) =
            *reinterpret_cast<const uint4 *>(a0.k + (int64_t(row) * a0.cap + j) * D + part * 8);
        if (part == 0) own_vl[j] = static_cast<const float *>(st.s_vlen)[srow + j];
      }
    }
  }
  __syncthreads();

  // Raw rows of update i: token p * RPP + sub of the thread's pass p, keys or
  // values, and the tokens' gates.
  uint4 raw[NP];
  uint16_t rg[NP];
  auto load_keys = [&](int i) __attribute__((always_inline)) {
    const int64_t tb = tok_lds[i];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int t = p * RPP + sub;
      if (p * RPP < n_tok) {
        const int64_t tt = tb + (t < n_tok ? t : 0);
        raw[p] = ld_stream16(k_row + tt * src.k_st + part * 8);
        rg[p] = g_row[tt * src.g_st];
      }
    }
  };
  // Token groups of 16 TT (a power of two of them) x slot groups fill the waves.
  int ntg = 1;
  while (ntg * (16 * TT) < n_tok) ntg <<= 1;
  const int nsg = kRowWaves / ntg, tg = wave % ntg, sg = wave / ntg;

  load_keys(0);
  for (int i = 0; i < list.count; ++i) {
    const int64_t u = int64_t(list.u0) + i;
    KVM_TS_A(0);
    // ---- prep (model/kvm_mixer.py:120-129, model/kvm_triton_mixer.py:429-446)
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      if (p * RPP < n_tok) {
        const int t = p * RPP + sub;
        float k[8];
        unpack8(raw[p], k);
        prep_key<D>(k, part, L, ln_w, ln_b);
        const float g = bf2f(rg[p]);
#pragma unroll
        for (int e = 0; e < 8; ++e) k[e] = L.gate_keys ? k[e] * g : k[e];
        *reinterpret_cast<uint4 *>(&tok[t * STR + part * 8]) = pack8(k);
        __builtin_amdgcn_sched_barrier(0);  // one pass at a time (register pressure)
      }
    }
    __syncthreads();

    KVM_TS_A(1);
    // ---- route (model/kvm_fp32_routing_reference.py:30-34)
    if (tg * (16 * TT) < n_tok) {
      uint4 bx[TT][KS];
#pragma unroll
      for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          bx[tt][ks] = *reinterpret_cast<const uint4 *>(
              &tok[(tg * (16 * TT) + tt * 16 + (lane & 15)) * STR + ks * 32 + (lane >> 4) * 8]);
      float best[TT];
      int bidx[TT];
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        best[tt] = -INFINITY;
        bidx[tt] = -1;
      }
      for (int blk = sg; blk < nblk; blk += nsg) {
        const int jb = blk * 16;
        uint4 a[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          a[ks] = *reinterpret_cast<const uint4 *>(&own_k[(jb + (lane & 15)) * STR + ks * 32 + (lane >> 4) * 8]);
        f32x4 accs[TT];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) accs[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int tt = 0; tt < TT; ++tt)
            accs[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[ks]), as_bf16x8(bx[tt][ks]), accs[tt], 0,
                                                               0, 0);
        const int j0 = jb + (lane >> 4) * 4;
        if (needs_scan(a[0], jb, protect, S)) {
#pragma unroll
          for (int tt = 0; tt < TT; ++tt) scan_max4(accs[tt], j0, protect, S, best[tt], bidx[tt]);
        } else {
#pragma unroll
          for (int tt = 0; tt < TT; ++tt) keep_max4(accs[tt], j0, best[tt], bidx[tt]);
        }
      }
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        uint64_t key = bidx[tt] >= 0 ? route_key(best[tt], bidx[tt]) : 0;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const uint32_t hi = uint32_t(key >> 32), lo = uint32_t(key);
          const uint64_t other = r == 0 ? (uint64_t(xor16_lane(hi, lane)) << 32) | xor16_lane(lo, lane)
                                        : (uint64_t(xor32_lane(hi, lane)) << 32) | xor32_lane(lo, lane);
          key = other > key ? other : key;
        }
        if (lane < 16) scratch[(sg * ntg + tg) * (16 * TT) + tt * 16 + lane] = key;
      }
    }
    __syncthreads();

    KVM_TS_A(2);
    {  // the raw values, in flight through the lists and the keys
      __builtin_amdgcn_sched_barrier(0);
      const int64_t tb = tok_lds[i];
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int t = p * RPP + sub;
        if (p * RPP < n_tok) raw[p] = ld_stream16(v_row + (tb + (t < n_tok ? t : 0)) * src.v_st + part * 8);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- lists: thread t has token t.
    uint64_t key = 0;
    if (tid < n_tok)
      for (int x = 0; x < nsg; ++x) {
        const uint64_t o = scratch[x * (ntg * 16 * TT) + tid];
        key = o > key ? o : key;
      }
    const int slot = route_key_slot(key);
    if (tid < n_tok) {
      const int64_t lo = u * log_stride + int64_t(row) * n_tok + tid;
      if (route_log) route_log[lo] = slot;
      if (append_log) append_log[lo] = 0;
    }
    __syncthreads();  // the route keys have been read; their place takes the counts
    const bool has = slot >= 0;
    uint64_t eq = __ballot(has);
    if (wave < LW)
#pragma unroll
      for (int x = 0; x < MAX; x += 64) wsc[wave * MAX + x + lane] = 0;
#pragma unroll
    for (int bit = 0; (1 << bit) < MAX; ++bit) {
      const uint64_t m = __ballot(has && ((slot >> bit) & 1));
      eq &= ((slot >> bit) & 1) ? m : ~m;
    }
    const int rank = int(__builtin_amdgcn_mbcnt_hi(uint32_t(eq >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(eq), 0u)));
    if (has && rank == 0) wsc[wave * MAX + slot] = uint16_t(__popcll(eq));
    __syncthreads();
    // Exclusive prefix: over the waves of each slot's counts (in place), then over the slots.
    int tot = 0;
    if (tid < MAX)
#pragma unroll
      for (int w = 0; w < LW; ++w) {
        const int c = wsc[w * MAX + tid];
        wsc[w * MAX + tid] = uint16_t(tot);
        tot += c;
      }
    int incl = tot;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o);
      if (lane >= o) incl += y;
    }
    if (lane == 63) wtot[wave] = incl;
    __syncthreads();
    {
      int base = incl - tot;
#pragma unroll
      for (int w = 0; w < LW; ++w) base += w < wave ? wtot[w] : 0;
      if (tid < MAX) {
        off[tid] = uint16_t(base);
        cnt[tid] = uint16_t(tot);
      }
    }
    __syncthreads();
    if (has) sorted[off[slot] + wsc[wave * MAX + slot] + rank] = uint16_t(tid);
    __syncthreads();

    KVM_TS_A(3);
    // Sum of the staged rows of slot j's tokens, in token order; whether there are any.
    auto sum_rows = [&](int j, float (&x)[8]) __attribute__((always_inline)) {
      const int n = j < S ? cnt[j] : 0, o = n > 0 ? off[j] : 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = 0.f;
      int e0 = 0;
      for (; e0 + 4 <= n; e0 += 4) {  // four rows' reads in flight
        uint4 r[4];
#pragma unroll
        for (int w = 0; w < 4; ++w)
          r[w] = *reinterpret_cast<const uint4 *>(&tok[int(sorted[o + e0 + w]) * STR + part * 8]);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          float f[8];
          unpack8(r[w], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] += f[e];
        }
      }
      for (; e0 < n; ++e0) {
        float f[8];
        unpack8(*reinterpret_cast<const uint4 *>(&tok[int(sorted[o + e0]) * STR + part * 8]), f);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] += f[e];
      }
      return n > 0;
    };
    const AttnRows nxt = snap_at(snaps, u + 1);
    const __amdgpu_buffer_rsrc_t nk = l2_rsrc(nxt.k + int64_t(row) * nxt.cap * D, int64_t(S) * D * 2);
    const __amdgpu_buffer_rsrc_t nv = l2_rsrc(nxt.v + int64_t(row) * nxt.cap * D, int64_t(S) * D * 2);
    const bool fin = i + 1 == list.count && list.final_rows != 0;

    // ---- keys (model/kvm_mixer.py:329-335): state = bf16(state + bf16(sum)),
    // LayerNorm.  Rows past S lie past the snapshot's resource and are not stored.
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      if (p * RPP < S) {
        const int j = p * RPP + sub;
        float x[8];
        const bool any = sum_rows(j, x);
        uint4 kk;
        if (__any(any)) {
          float k[8];
          unpack8(sk[p], k);
          if (any) {
            round_pack8(x);
#pragma unroll
            for (int e = 0; e < 8; ++e) k[e] += x[e];
            sk[p] = round_pack8(k);
          }
          layer_norm8<D>(k, part, ln_w, ln_b, float(L.ln_eps));
          kk = pack8(k);
          if (j < S) *reinterpret_cast<uint4 *>(&own_k[j * STR + part * 8]) = kk;
        } else {  // no slot of this wave's pass changed
          kk = *reinterpret_cast<const uint4 *>(&own_k[j * STR + part * 8]);
        }
        st16<kPolicyNT>(nk, uint32_t((j * D + part * 8) * 2), kk);
        if (fin && j < S) *reinterpret_cast<uint4 *>(s_ka + (srow + j) * D + part * 8) = kk;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();  // every wave has read the merge keys
    KVM_TS_A(4);
    // ---- values
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      if (p * RPP < n_tok) {
        float v[8];
        unpack8(raw[p], v);
        const float g = bf2f(rg[p]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = L.gate_values ? v[e] * g : v[e];
        *reinterpret_cast<uint4 *>(&tok[(p * RPP + sub) * STR + part * 8]) = pack8(v);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (i + 1 < list.count) load_keys(i + 1);
    __syncthreads();
    KVM_TS_A(5);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      if (p * RPP < S) {
        const int j = p * RPP + sub;
        float x[8], v[8];
        const bool any = sum_rows(j, x);
        unpack8(sv[p], v);
        if (any) {
          round_pack8(x);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += x[e];
          sv[p] = round_pack8(v);
        }
        const uint4 vv = attn_value8_packed<D>(v, j < S ? own_vl[j] : 0.f);
        st16<kPolicyNT>(nv, uint32_t((j * D + part * 8) * 2), vv);
        if (fin && j < S) *reinterpret_cast<uint4 *>(s_va + (srow + j) * D + part * 8) = vv;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();  // every wave has read the merge values
    KVM_TS_A(6);
  }
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int j = p * RPP + sub;
    if (j < S) {
      *reinterpret_cast<uint4 *>(s_k + (srow + j) * D + part * 8) = sk[p];
      *reinterpret_cast<uint4 *>(s_v + (srow + j) * D + part * 8) = sv[p];
    }
  }
}

__global__ __launch_bounds__(256) void k_fill_u32(unsigned *p, int64_t n, unsigned v) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}

}  // namespace

namespace {
// Rows of G members that one launch keeps resident: one group per XCD at a
// time, so whole eights.  0 where the device does not hold eight groups.
int rows_per_launch(int64_t limit, int G) { return int(limit / G / 8 * 8); }
}  // namespace

bool chain_plan(const kvm_layer &L, int64_t n_tok, int64_t max_slots, ChainPlan *p) {
  int dev = 0, cus = 0;
  return hipGetDevice(&dev) == hipSuccess &&
         hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
         chain_plan_on(cus, L, n_tok, max_slots, p);
}

bool chain_plan_on(int64_t cus, const kvm_layer &L, int64_t n_tok, int64_t max_slots, ChainPlan *p) {
  // Every member of a group must be resident at once: at most one
  // workgroup per compute unit.
  const int64_t limit = std::min<int64_t>(kChainMaxWorkgroups, cus);
  const int64_t rows = L.batch * L.kv_heads;
  const int64_t groups = (rows + 7) / 8 * 8;
  // Members per row of the appending chain: 16 while every row fits one
  // launch, 8 up to what that keeps resident, then 4 (each launch holds twice
  // the rows of 8 members and takes less than twice as long: us per update for
  // all rows with 8 / 4 members, 48 rows of 1425 slots 57.0 / 38.8, 64 rows of
  // 872 64-wide slots 38.3 / 23.6, 256 rows of 868 slots, C 128, 190 / 116).
  // More rows than a launch keeps resident: consecutive launches over batches
  // of rows (launch_chain).
  for (int G : {16, 4, 8}) {
    if ((G == 16 && groups * 16 > limit) || (G == 4 && groups * 8 <= limit)) continue;
    const int64_t tpw = ((n_tok + G - 1) / G + 15) / 16 * 16;
    const int64_t own_cap = ((max_slots + 15) / 16 + G - 1) / G * 16;
    if (tpw > kChainTok || rows_per_launch(limit, G) == 0 || n_tok < 1 || max_slots > 65536) continue;
    const int64_t dyn = append_lds_bytes(int(n_tok), int(own_cap));
    if (dyn > kAppendDynLds) continue;
    p->fixed = false;
    p->G = G;
    p->limit = int(limit);
    p->rows = int(rows);
    p->head_dim = int(L.head_dim);
    p->tpw = int(tpw);
    p->own_cap = int(own_cap);
    p->dyn_lds = size_t(dyn);
    return true;
  }
  return false;
}

namespace {
// Members per row of a chain without appends over S slots (1: k_chain_row),
// or 0 when none fits.  Up to 16 rows: 16 members (chain_plan).  Above, more
// members make an update shorter but fewer rows fit a launch, so the choice
// is the least of launches x time per update.  Measured, us per update for all
// rows, with 8 / 4 / 1 members (24 and 40 rows fill one launch of 8 and of 4):
//   D    C    S     24 rows             40 rows              96 rows             256 rows
//   128  256  256    7.8 /  9.8 / 21.1   15.0 / 10.1 / 22.0   23.7 / 20.5 / 22.7  63.5 / 47.8 / 30.6
//   128  128  256    7.2 /  8.6 / 16.4   13.8 /  8.7 / 16.7   22.4 / 18.4 / 17.7  56.2 / 35.4 / 22.9
//   128   64  256    6.9 /  8.1 / 13.7   13.1 /  8.4 / 13.9   20.4 / 17.1 / 14.8  52.0 / 33.4 / 16.6
//   128  128  128    6.4 /  7.0 / 12.4   12.7 /  7.0 / 12.3   19.6 / 14.5 / 13.0  51.6 / 29.2 / 16.7
//   128   16   16    5.8 /  5.6 /  6.7   11.5 /  5.7 /  6.7   17.5 / 11.5 /  6.9  45.7 / 23.1 /  7.0
//    64  256  256    5.6 /  6.7 / 14.4   11.5 /  6.9 / 14.0   17.9 / 14.0 / 14.7  46.9 / 28.3 / 16.8
//    64  128  512    6.2 /  8.7 / 15.6   12.3 /  8.9 / 15.5   19.0 / 18.1 / 16.7  49.5 / 35.4 / 17.1
//    64  128  128    4.4 /  5.2 /  8.7   10.5 /  5.3 /  8.8   15.3 / 10.8 /  8.7  42.0 / 22.3 /  9.5
//    64   16   16    4.7 /  4.4 /  6.3    9.4 /  4.7 /  6.6   14.4 /  9.4 /  6.6  37.8 / 18.8 /  6.7
//    64  512  512    8.0 /   -  / 28.3   15.8 /   -  / 29.1   25.9 /   -  / 30.2  69.0 /   -  / 34.8
// (C 512: 4 members would prep 128 tokens each, which their staging rows do
// not hold.)  The lines below fit these and 18 more shapes: a part that is
// latency, and parts that grow with the tokens and slots a member works on.
int fixed_group(const ChainPlan &p, int S, int64_t n_tok) {
  if (n_tok > kFixedMaxTok) return 0;
  const int nblk = (S + 15) / 16;
  // Owned slots per member: up to 64 at G = 16, up to 128 below; at most kChainTok prep tokens;
  // and a launch that holds eight groups, which the plan has checked for its own G only.
  const auto fits = [&](int G) {
    return rows_per_launch(p.limit, G) > 0 && (nblk + G - 1) / G * 16 <= (G == 16 ? 64 : kOwnMax) &&
           (n_tok + G - 1) / G <= kChainTok;
  };
  if (p.G == 16) return fits(16) ? 16 : 0;
  const bool wide = p.head_dim == 128;
  const double tok = double(n_tok) * p.head_dim / 128, slots = double(S) * p.head_dim / 128;
  const auto launches = [&](int G) {
    const int per = G == 1 ? p.limit : rows_per_launch(p.limit, G);
    return double((p.rows + per - 1) / per);
  };
  int best = 0;
  double least = 0;
  const auto offer = [&](int G, double us) {
    if (best == 0 || us < least) {
      best = G;
      least = us;
    }
  };
  const int rmax = wide ? RowMax<128>::value : RowMax<64>::value;
  if (fits(8)) offer(8, launches(8) * ((wide ? 5.2 : 4.2) + 0.0066 * (tok + slots)));
  if (fits(4)) offer(4, launches(4) * ((wide ? 4.7 : 4.2) + 0.0125 * (tok + slots)));
  if (S <= rmax && n_tok <= rmax) offer(1, launches(1) * (5.2 + 0.05 * tok + 0.026 * slots));
  return best;
}
}  // namespace

bool chain_fixed_ok(const ChainPlan &p, const ChainList &list, int64_t n_tok) {
  if (list.count < 1) return false;
  const int S = list.state_before[0];
  for (int i = 0; i < list.count; ++i)
    if (list.n_append[i] != 0 || list.state_before[i] != S) return false;
  return fixed_group(p, S, n_tok) != 0;
}

void chain_shape(const ChainPlan &p, int64_t state_len, int64_t n_tok, int32_t *shape) {
  const int G = state_len >= 1 && state_len <= 0x7fff ? fixed_group(p, int(state_len), n_tok) : 0;
  shape[0] = p.G;
  shape[1] = rows_per_launch(p.limit, p.G);
  shape[2] = G;
  shape[3] = G == 0 ? 0 : G == 1 ? p.rows : rows_per_launch(p.limit, G);
}

int64_t chain_scratch_bytes(const kvm_layer &L, int64_t n_tok) {
  const size_t tok = size_t(L.batch * L.kv_heads) * size_t(n_tok);
  auto a256 = [](size_t x) { return (x + 255) & ~size_t(255); };
  // four merge buffers of keys, four of values (buffer b at gk + b * rows * n_tok * D),
  // per-member novelties and two sets of route maxima (up to 16 members), counters
  return int64_t(2 * a256(4 * tok * size_t(L.head_dim) * 2) + a256(tok * 16 * 4) +
                 a256(2 * tok * 16 * 8) +
                 a256(size_t(kChainMaxWorkgroups) * kCounterStride * 4 + 256));
}

ChainScratch carve_chain_scratch(void *base, const kvm_layer &L, int64_t n_tok) {
  const size_t tok = size_t(L.batch * L.kv_heads) * size_t(n_tok);
  auto a256 = [](size_t x) { return (x + 255) & ~size_t(255); };
  unsigned char *p = static_cast<unsigned char *>(base);
  ChainScratch c;
  const size_t kb = tok * size_t(L.head_dim) * 2, ib = a256(tok * 16 * 4);
  const size_t kb4 = a256(4 * kb), pb = a256(2 * tok * 16 * 8);
  c.gk = reinterpret_cast<uint16_t *>(p);
  c.gv = reinterpret_cast<uint16_t *>(p + kb4);
  c.nov = reinterpret_cast<float *>(p + 2 * kb4);
  c.part = reinterpret_cast<uint2 *>(p + 2 * kb4 + ib);
  c.bar = reinterpret_cast<unsigned *>(p + 2 * kb4 + ib + pb);
  c.abort_flag = c.bar + size_t(kChainMaxWorkgroups) * kCounterStride;
  c.status = nullptr;  // set by the caller
  c.max_polls = kChainDefaultPolls;
  return c;
}

hipError_t launch_fill_u32(unsigned *p, int64_t n, unsigned v, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u32, dim3(unsigned((n + 255) / 256)), dim3(256), 0, stream, p, n, v);
  return hipGetLastError();
}

hipError_t launch_chain(const kvm_layer &L, const kvm_seq &src, int64_t n_tok,
                        const kvm_state &st, const SnapRing &snaps, const ChainList &list,
                        const ChainScratch &cs, const ChainPlan &p, int32_t *route_log,
                        int32_t *append_log, hipStream_t stream) {
  if (list.count <= 0) return hipSuccess;
  const int rows = int(L.batch * L.kv_heads);
  const int64_t log_stride = int64_t(rows) * n_tok;
  const bool fixed = p.fixed && chain_fixed_ok(p, list, n_tok);
  const int G = fixed ? fixed_group(p, list.state_before[0], n_tok) : p.G;
  if (G == 1) {  // one independent workgroup per row
    if (L.head_dim == 128)
      hipLaunchKernelGGL(k_chain_row<128>, dim3(unsigned(rows)), dim3(kRowThreads), 0, stream, L, src, int(n_tok),
                         st, snaps, list, route_log, append_log, log_stride);
    else
      hipLaunchKernelGGL(k_chain_row<64>, dim3(unsigned(rows)), dim3(kRowThreads), 0, stream, L, src, int(n_tok),
                         st, snaps, list, route_log, append_log, log_stride);
    return hipGetLastError();
  }
  const int row_batch = rows_per_launch(p.limit, G);
  if (row_batch <= 0) return hipErrorInvalidConfiguration;
  for (int row0 = 0; row0 < rows; row0 += row_batch) {
    const int nrows = std::min(row_batch, rows - row0);
    // Barrier counters and the abort flag start at zero in every launch.
    hipError_t e = launch_fill_u32(cs.bar, kChainMaxWorkgroups * kCounterStride + 64, 0u, stream);
    if (e != hipSuccess) return e;
    const dim3 grid(unsigned((nrows + 7) / 8 * 8 * G)), blk(kChainThreads);
    if (fixed) {
      const int nt = int(n_tok);
      const bool own128 = ((list.state_before[0] + 15) / 16 + G - 1) / G * 16 > 64;  // G < 16 then
#define KVM_FIXED(DD, GG, OO)                                                                               \
  hipLaunchKernelGGL((k_chain_fixed<DD, GG, OO>), grid, blk, 0, stream, L, src, nt, st, snaps, list, cs, rows, \
                     row0, nrows, route_log, append_log, log_stride)
#define KVM_FIXED_D(DD)            \
  if (G == 16)                     \
    KVM_FIXED(DD, 16, 64);         \
  else if (G == 8 && own128)       \
    KVM_FIXED(DD, 8, 128);         \
  else if (G == 8)                 \
    KVM_FIXED(DD, 8, 64);          \
  else if (own128)                 \
    KVM_FIXED(DD, 4, 128);         \
  else                             \
    KVM_FIXED(DD, 4, 64)
      if (L.head_dim == 128) {
        KVM_FIXED_D(128);
      } else {
        KVM_FIXED_D(64);
      }
#undef KVM_FIXED_D
#undef KVM_FIXED
    } else {
#define KVM_APPEND(DD, GG)                                                                                   \
  hipLaunchKernelGGL((k_chain<DD, GG>), grid, blk, p.dyn_lds, stream, L, src, int(n_tok), st, snaps, list, cs, \
                     rows, row0, nrows, p.tpw, p.own_cap, route_log, append_log, log_stride)
#define KVM_APPEND_D(DD)   \
  if (G == 16)             \
    KVM_APPEND(DD, 16);    \
  else if (G == 8)         \
    KVM_APPEND(DD, 8);     \
  else                     \
    KVM_APPEND(DD, 4)
      if (L.head_dim == 128) {
        KVM_APPEND_D(128);
      } else {
        KVM_APPEND_D(64);
      }
#undef KVM_APPEND_D
#undef KVM_APPEND
    }
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace kvm

#ifdef KVM_CHAIN_TIMING
// Copies the phase timestamps (2 x 128 x 16 words) of the last timed launch.
extern "C" int kvm_chain_timing_read(void *dst, long words) {
  return int(hipMemcpyFromSymbol(dst, HIP_SYMBOL(kvm::g_chain_ts), size_t(words) * 8));
}
#endif
