// ILU(0) preconditioner on gfx950: factorisation and triangular sweeps
// (PRECO_ILU0::Factor / Solve, Preco_ilu0.cpp:64-186, 497-530, 958-980).
//
// An Ilu object holds one ILU(0) system: the CSR pattern, the schedule of its factorisation,
// the packed sweep layouts, and FP64 / FP32 factors.  Both instances of a context factor the
// whole matrix in the reference's equation order (its FP32 factors are bit-identical to the
// reference's); they differ in the sweeps:
//  * the reference sweeps: the whole lower / upper factor (the plain FP64 path);
//  * strip sweeps: rows are cut into contiguous ranges (the frontal order runs along the
//    channel, so a range is a strip of cross-sections), strips into blocks, and the factor
//    entries that couple two blocks are left out of the sweeps, so blocks are swept apart.
//    The pivots stay those of the full factorisation (factoring the strips separately
//    loses the upstream couplings at each strip start and leaves near-zero pivots).
//    It preconditions the FP32 solve inside the FP64 refinement, where the FP64 residual,
//    not the preconditioner, decides the answer.
//
// Factorisation: one persistent launch, one wave per unit of up to three rows (k_unit_flow), or
// per row where the pattern does not allow that (a row with a column twice among them) and after a
// pivot repair (k_ilu_flow); row i
// eliminates its lower entries in increasing column order, so every factor entry gets its
// updates in the reference's order and, with FMA contraction off, the reference's
// rounding.  Multipliers are stored negated as in the reference.
//
// Sweeps: blocks of at most BS_ROWS rows by a wave each with their values in LDS: of the strip
// sweeps 16 rows at a time (k_chunk_sweep), of many blocks or in the reference order level by
// level (k_block_sweep); others by a workgroup per strip that walks the levels of nodes, LDS holding
// the rows that later levels still read (k_node_sweep); where those do not fit LDS, or a row has a
// column twice, the staged level sweep (k_sweep_stage), whose values go through an LDS ring of RING positions and a
// global copy in processing order: a level reads a dependency from the ring while its slot has
// not been reused (position >= P + nr - RING for a level of nr rows starting at P) and from the
// global copy otherwise, which is safe because a full barrier (global release / acquire) is
// taken whenever the position crosses a multiple of FENCE, and any value that has left the ring
// is older than the last such barrier (nr <= RING/4).  Wider levels read everything from the
// global copy between full barriers.
#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <future>
#include <type_traits>

#include "rmx_internal.h"

namespace rmx {

constexpr int FW = 128;         // maximum row width handled by the factorisation
constexpr int LPC = 1024;       // level offsets staged in LDS at a time
constexpr int FENCE = 2048;     // positions between full barriers
constexpr int WIDE = RING / 4;  // levels wider than this use the global copy only
constexpr int STAGE_THREADS = 512;                 // staged sweep: threads per workgroup
constexpr int STAGE_ROWS = STAGE_THREADS / 4;      // rows per round (4 lanes per row)

// ---------------------------------------------------------------------------------------
// factorisation

constexpr int UCAP = 2048;      // entries of the pivot rows staged in LDS per row
constexpr int UPL = UCAP / 64;  // staged entries per lane

// One row of one level (one wave): row i eliminates its lower entries k in increasing
// column order (IKJ).  Per-pattern metadata keeps the dependent memory rounds to three: the
// row's descriptor {i, start, width, lower count}; the row (values, sorted columns) with
// the start and length of every pivot row; then all pivot rows at once, staged in LDS with
// independent loads, every staged entry getting its target position in row i (a binary
// search over row i's sorted columns, done in parallel).  The sequential loop over k is
// then one division and one LDS update per entry.  The updates are the reference's, in its
// order, with FMA contraction off.  Rows whose pivot rows hold more than UCAP entries
// search and read from global memory inside the loop instead.
// Symbolic plan of the factorisation (once per pattern, all rows in one launch, one wave
// per row): every entry u of a row's concatenated pivot rows (the entries after each pivot
// row's diagonal, in sorted lower-column order of the row) gets its pivot index t (low
// byte) and its target position in the row (high byte; 255: not in the row, or a column at
// or left of the pivot).
__global__ void __launch_bounds__(64) k_ilu_plan(const int4* __restrict__ desc, int cnt,
                                                 const int* __restrict__ cols,
                                                 const int* __restrict__ srt_cols,
                                                 const unsigned char* __restrict__ srt_pos,
                                                 const int2* __restrict__ piv,
                                                 const long long* __restrict__ pbase,
                                                 unsigned short* __restrict__ plan)
{
  __shared__ int s_col[FW], s_kb[FW], s_off[FW + 1];
  __shared__ unsigned char s_pos[FW];
  const int lane = threadIdx.x;
  const int w = blockIdx.x;
  if (w >= cnt) return;
  const int4 d = desc[w];
  const int p0 = d.y, wi = d.z, nk = d.w;
  for (int t = lane; t < wi; t += 64) {
    s_col[t] = srt_cols[p0 + t];
    s_pos[t] = srt_pos[p0 + t];
  }
  int carry = 0;
  for (int t0 = 0; t0 < nk; t0 += 64) {
    const int t = t0 + lane;
    int len = 0;
    if (t < nk) {
      const int2 pv = piv[p0 + t];
      s_kb[t] = pv.x;
      len = pv.y;
    }
    int incl = len;
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    if (t < nk) s_off[t + 1] = carry + incl;
    carry += __shfl(incl, 63, 64);
  }
  if (lane == 0) s_off[0] = 0;
  __syncthreads();
  const int total = s_off[nk];
  const long long pb = pbase[w];
  for (int u = lane; u < total; u += 64) {
    int lo = 0, hi = nk - 1;                // pivot t with s_off[t] <= u < s_off[t+1]
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s_off[mid] <= u) lo = mid; else hi = mid - 1;
    }
    const int k = s_col[lo];
    const int cc = cols[s_kb[lo] + 1 + (u - s_off[lo])];
    int pos = 255;
    if (cc > k) {
      int a = 0, b = wi - 1;
      while (a <= b) {
        const int mid = (a + b) >> 1;
        const int v = s_col[mid];
        if (v == cc) { pos = s_pos[mid]; break; }
        if (v < cc) a = mid + 1; else b = mid - 1;
      }
    }
    plan[pb + u] = (unsigned short)(lo | (pos << 8));
  }
}

// Staged pivot-row entries of one row, in rounds of 64 (entry u = lane + 64 m) grouped in
// chunks of PCH rounds: a chunk is taken when the row has entries in it (a wave-uniform
// test), and inside a chunk no lane branches around a load (lanes past the last entry read
// it again), so a chunk's loads are all issued before the first wait.  plan_offsets: the
// target position of every entry and the offset (from element base) of its value in its
// pivot row; stage_entries: the loaded values and targets into LDS.
constexpr int PCH = 8;
__device__ __forceinline__ void plan_offsets(const unsigned short* __restrict__ plan, int total,
                                             const int* s_kb, const int* s_off, int base,
                                             unsigned* offs, unsigned char* pp)
{
  const int lane = threadIdx.x;
  unsigned short tp[UPL];
#pragma unroll
  for (int c = 0; c < UPL / PCH; c++)
    if (c * PCH * 64 < total) {
#pragma unroll
      for (int m = c * PCH; m < (c + 1) * PCH; m++) tp[m] = plan[min(lane + 64 * m, total - 1)];
#pragma unroll
      for (int m = c * PCH; m < (c + 1) * PCH; m++) {
        const int u = min(lane + 64 * m, total - 1);
        const int t = tp[m] & 0xFF;
        pp[m] = (unsigned char)(tp[m] >> 8);
        offs[m] = (unsigned)(s_kb[t] - base + 1 + (u - s_off[t]));
      }
    }
}

template <class VT>
__device__ __forceinline__ void stage_entries(int total, const unsigned* offs,
                                              const unsigned char* pp, const VT* uv,
                                              unsigned char* s_upos, VT* s_uval)
{
  const int lane = threadIdx.x;
#pragma unroll
  for (int c = 0; c < UPL / PCH; c++)
    if (c * PCH * 64 < total) {
#pragma unroll
      for (int m = c * PCH; m < (c + 1) * PCH; m++) {
        const int u = lane + 64 * m;
        if (u < total) {
          s_upos[u] = pp[m];
          s_uval[u] = uv[m];
        }
      }
    }
}

template <class VT>
__global__ void __launch_bounds__(64) k_ilu_level(const int4* __restrict__ desc, int cnt,
                                                  const int* __restrict__ cols,
                                                  const int* __restrict__ srt_cols,
                                                  const unsigned char* __restrict__ srt_pos,
                                                  const int2* __restrict__ piv,
                                                  const long long* __restrict__ pbase,
                                                  const unsigned short* __restrict__ plan,
                                                  VT* __restrict__ LU, int* __restrict__ err,
                                                  const int4* __restrict__ desc_next,
                                                  int cnt_next,
                                                  const long long* __restrict__ pbase_next,
                                                  long long plan_n)
{
#pragma clang fp contract(off)
  __shared__ VT s_val[FW];
  __shared__ int s_col[FW];
  __shared__ unsigned char s_pos[FW];
  __shared__ int s_kb[FW], s_off[FW + 1];
  __shared__ VT s_dk[FW];
  __shared__ unsigned char s_upos[UCAP];
  __shared__ VT s_uval[UCAP];
  const int lane = threadIdx.x;
  const int w = blockIdx.x;
  if (w >= cnt) return;                 // uniform per block
  const int4 d = desc[w];
  const int i = d.x, p0 = d.y, wi = d.z, nk = d.w;
  // the next level's row at this index: its descriptor now, its static data (and initial
  // values, which no other row writes) touched after this row's own loads are issued, so
  // the next launch finds them in the memory-side cache
  const bool pre = w < cnt_next;
  int4 dn = make_int4(0, 0, 0, 0);
  long long pbn = 0;
  if (pre) { dn = desc_next[w]; pbn = pbase_next[w]; }
  for (int t = lane; t < wi; t += 64) {
    s_val[t] = LU[p0 + t];
    s_col[t] = srt_cols[p0 + t];
    s_pos[t] = srt_pos[p0 + t];
  }
  // pivot rows (the first nk sorted columns): start and entries after the diagonal;
  // offsets of their staged entries by an inclusive wave scan
  int carry = 0;
  for (int t0 = 0; t0 < nk; t0 += 64) {
    const int t = t0 + lane;
    int len = 0;
    if (t < nk) {
      const int2 pv = piv[p0 + t];
      s_kb[t] = pv.x;
      len = pv.y;
    }
    int incl = len;
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    if (t < nk) s_off[t + 1] = carry + incl;
    carry += __shfl(incl, 63, 64);
  }
  if (lane == 0) s_off[0] = 0;
  __syncthreads();
  // target position in row i of a column cc of pivot row k (255: not in row i, or cc <= k)
  auto target = [&](int cc, int k) -> int {
    if (cc <= k) return 255;
    int lo = 0, hi = wi - 1;
    while (lo <= hi) {
      const int mid = (lo + hi) >> 1;
      const int v = s_col[mid];
      if (v == cc) return s_pos[mid];
      if (v < cc) lo = mid + 1; else hi = mid - 1;
    }
    return 255;
  };
  const int total = s_off[nk];
  const bool staged = total <= UCAP;
  for (int t = lane; t < nk; t += 64) s_dk[t] = LU[s_kb[t]];
  if (staged) {                         // pivot-row values, targets from the plan
    const long long pb = pbase[w];
    unsigned offs[UPL];
    unsigned char pp[UPL];
    plan_offsets(plan + pb, total, s_kb, s_off, 0, offs, pp);
    VT uv[UPL];
#pragma unroll
    for (int c = 0; c < UPL / PCH; c++)
      if (c * PCH * 64 < total) {
#pragma unroll
        for (int m = c * PCH; m < (c + 1) * PCH; m++) uv[m] = LU[offs[m]];
      }
    stage_entries(total, offs, pp, uv, s_upos, s_uval);
  }
  unsigned int sink = 0;
  if (pre) {
    for (int t = lane; t < dn.z; t += 64)
      sink += (unsigned int)srt_cols[dn.y + t] + (unsigned int)srt_pos[dn.y + t] +
              (unsigned int)(LU[dn.y + t] != (VT)0);
    for (int t = lane; t < dn.w; t += 64) sink += (unsigned int)piv[dn.y + t].x;
    for (long long u = pbn + 128LL * lane; u < pbn + UCAP && u < plan_n; u += 128LL * 64)
      sink += (unsigned int)plan[u];
  }
  __syncthreads();
  if (staged) {
    // pivot t's diagonal position and value and this lane's (at most two) entries of its
    // pivot row (target, value) are read one pivot ahead, so that a pivot's chain is the
    // read of the two row values, the division and the update
    auto load_piv = [&](int t, int& pik, VT& dk, int& pa, VT& ua, int& pb, VT& ub_) {
      pik = s_pos[t];
      dk = s_dk[t];
      const int lo = s_off[t], hi = s_off[t + 1];
      const int e0 = lo + lane, e1 = e0 + 64;
      pa = 255; pb = 255; ua = (VT)0; ub_ = (VT)0;
      if (e0 < hi) { pa = s_upos[e0]; ua = s_uval[e0]; }
      if (e1 < hi) { pb = s_upos[e1]; ub_ = s_uval[e1]; }
    };
    int pik = 0, pa = 255, pb = 255;
    VT dk = (VT)1, ua = (VT)0, ub_ = (VT)0;
    if (nk > 0) load_piv(0, pik, dk, pa, ua, pb, ub_);
    for (int t = 0; t < nk; t++) {
      int pikn = 0, pan = 255, pbn = 255;
      VT dkn = (VT)1, uan = (VT)0, ubn = (VT)0;
      if (t + 1 < nk) load_piv(t + 1, pikn, dkn, pan, uan, pbn, ubn);
      const VT a = s_val[pik];
      const VT ca = pa != 255 ? s_val[pa] : (VT)0;
      const VT cb = pb != 255 ? s_val[pb] : (VT)0;
      const VT f = -a / dk;                // every lane, from the same LDS values
      if (pa != 255) { const VT prod = f * ua; s_val[pa] = ca + prod; }
      if (pb != 255) { const VT prod = f * ub_; s_val[pb] = cb + prod; }
      __syncthreads();                    // the updates before the next pivot
      if (lane == 0) s_val[pik] = f;      // the stored multiplier (no later pivot reads it)
      pik = pikn; dk = dkn; pa = pan; ua = uan; pb = pbn; ub_ = ubn;
    }
  } else {
    for (int t = 0; t < nk; t++) {
      const int k = s_col[t];
      const int pik = s_pos[t];
      const VT f = -s_val[pik] / s_dk[t];
      const int ua = s_off[t], ub = s_off[t + 1];
      for (int e = lane; e < ub - ua; e += 64) {
        const int q = s_kb[t] + 1 + e;
        const int pos = target(cols[q], k);
        if (pos != 255) {
          const VT prod = f * LU[q];
          s_val[pos] = s_val[pos] + prod;
        }
      }
      __syncthreads();                    // the stored multiplier and updates before the next k
      if (lane == 0) s_val[pik] = f;
    }
  }
  __syncthreads();
  for (int t = lane; t < wi; t += 64) LU[p0 + t] = s_val[t];
  if (lane == 0 && fabs((double)s_val[0]) < 1.0e-20) atomicOr(err, 1);
  if (sink == 0x9E3779B9u && cnt < 0) err[1] = (int)sink;   // keeps the touches (never taken)
}

// ---------------------------------------------------------------------------------------
// dataflow factorisation: one persistent launch instead of one launch per level

// Loads and stores of factor values that other waves of the same launch write or read are
// agent-scope atomics (sc1: coherent across the XCDs' L2 caches), and so are the row
// completion flags.  A row publishes its values, waits until they are performed
// (vmcnt(0): the stores are acknowledged at agent scope) and then stores its flag; a
// consumer issues its loads of a pivot row only after its flag load has returned the
// current epoch.  No cache-wide write-back or invalidate is needed.
__device__ __forceinline__ int ld_flag(const int* p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_flag(int* p, int v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Factor values through a buffer resource based at a wave-uniform element (32-bit byte
// offsets from it), with the sc1 cache policy: plain loads and stores, so the compiler
// batches them under one wait, and coherent at agent scope.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sc1_rsrc(const void* base)
{
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, -1, 0x00020000);
}
__device__ __forceinline__ float ld_sc1(__amdgpu_buffer_rsrc_t r, unsigned e, float)
{
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, e * 4u, 0, 16));
}
__device__ __forceinline__ double ld_sc1(__amdgpu_buffer_rsrc_t r, unsigned e, double)
{
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, e * 8u, 0, 16));
}
__device__ __forceinline__ void st_sc1(__amdgpu_buffer_rsrc_t r, unsigned e, float v)
{
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, e * 4u, 0, 16);
}
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void st_sc1(__amdgpu_buffer_rsrc_t r, unsigned e, double v)
{
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, e * 8u, 0, 16);
}

enum { FLOW_COUNTER = 0, FLOW_ERR = 1, FLOW_ABORT = 2, FLOW_BADROW = 3 };

// Ordering of LDS accesses inside one wave: a one-wave workgroup needs no barrier (a wave's
// LDS operations complete in order); the fences keep the compiler from moving accesses
// across it.
__device__ __forceinline__ void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Waves take rows in level order from a counter (one device-scope fetch-add per row, about
// 12 ns on this part).  A pivot row is earlier in that order than the rows that need it, so
// it has been taken by a running wave and every wait ends; no wave has to be resident
// before it takes work.  Per row: the row's own values, its sorted columns and plan are
// read with plain loads (no other wave writes them).  The pivots are then eliminated in
// increasing column order, as the reference does (update order kept, FMA contraction off),
// progressively: the run of pivots from the next one whose rows are done (one flag load
// per pivot) is staged and eliminated; when the next pivot's row is not done, one lane
// polls its flag (bounded by spin_limit polls, after which the row sets the abort flag
// that ends every wave's waits).  The rows finished last are usually the last pivots, so
// most of a row's work is done before its last pivot row arrives.  The finished row is
// stored and its flag set to the factorisation's epoch.  Rows whose pivot rows hold more
// entries than the LDS staging first wait for all their pivots and read the entries from
// memory.
template <class VT>
__global__ void __launch_bounds__(64) k_ilu_flow(const int4* __restrict__ desc, int n,
                                                 const int* __restrict__ cols,
                                                 const int* __restrict__ srt_cols,
                                                 const unsigned char* __restrict__ srt_pos,
                                                 const int2* __restrict__ piv,
                                                 const long long* __restrict__ pbase,
                                                 const unsigned short* __restrict__ plan,
                                                 VT* __restrict__ LU, int* __restrict__ done,
                                                 int epoch, int* __restrict__ state,
                                                 int spin_limit, int skip_upto)
{
#pragma clang fp contract(off)
  __shared__ VT s_val[FW];
  __shared__ int s_col[FW];
  __shared__ unsigned char s_pos[FW];
  __shared__ int s_kb[FW], s_off[FW + 1];
  __shared__ VT s_dk[FW];
  __shared__ unsigned char s_upos[UCAP];
  __shared__ VT s_uval[UCAP];
  const int lane = threadIdx.x;
  int polls = 0;
  // one lane polls the flag of row k until it holds the epoch; false: aborted
  auto wait_row = [&](int k) -> bool {
    for (;;) {
      int v = 0;
      if (lane == 0) v = ld_flag(done + k);
      if (__builtin_amdgcn_readfirstlane(v) == epoch) return true;
      if ((++polls & 31) == 0) {
        int ab = 0;
        if (lane == 0) ab = ld_flag(state + FLOW_ABORT);
        if (__builtin_amdgcn_readfirstlane(ab) != 0 || polls > spin_limit) return false;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  };
  for (;;) {
    int w = 0;
    if (lane == 0) w = __hip_atomic_fetch_add(state + FLOW_COUNTER, 1, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
    w = __builtin_amdgcn_readfirstlane(w);
    if (w >= n) break;
    const int4 d = desc[w];
    const int i = d.x, p0 = d.y, wi = d.z, nk = d.w;
    if (i <= skip_upto) continue;                  // final from an earlier pass
    for (int t = lane; t < wi; t += 64) {
      s_val[t] = LU[p0 + t];
      s_col[t] = srt_cols[p0 + t];
      s_pos[t] = srt_pos[p0 + t];
    }
    int carry = 0;
    for (int t0 = 0; t0 < nk; t0 += 64) {
      const int t = t0 + lane;
      int len = 0;
      if (t < nk) {
        const int2 pv = piv[p0 + t];
        s_kb[t] = pv.x;
        len = pv.y;
      }
      int incl = len;
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o, 64);
        if (lane >= o) incl += v;
      }
      if (t < nk) s_off[t + 1] = carry + incl;
      carry += __shfl(incl, 63, 64);
    }
    if (lane == 0) s_off[0] = 0;
    wave_sync();
    const int total = s_off[nk];
    const bool staged = total <= UCAP;
    // pivot rows lie within one band of rows: offsets from the first fit 32 bits
    const int kb0 = nk > 0 ? __builtin_amdgcn_readfirstlane(s_kb[0]) : p0;
    const __amdgpu_buffer_rsrc_t rp = sc1_rsrc(LU + kb0);
    bool aborted = false;
    polls = 0;
    if (staged) {
      unsigned offs[UPL];
      unsigned char pp[UPL];
      plan_offsets(plan + pbase[w], total, s_kb, s_off, kb0, offs, pp);
      int ta = 0;
      bool waited = false;                        // pivot ta's row was just seen done
      while (ta < nk) {
        // tb: the first pivot from ta on whose row is not done (after a wait: ta alone,
        // whose flag was read last, so its entries load without another flag round trip)
        int tb = ta + 1;
        if (!waited) {
          tb = nk;
          for (int t0 = ta; t0 < nk; t0 += 64) {
            const int t = t0 + lane;
            const bool ok = t >= nk || ld_flag(done + s_col[t]) == epoch;
            const unsigned long long pend = __ballot(!ok);
            if (pend) { tb = t0 + (int)__builtin_ctzll(pend); break; }
          }
          if (tb == ta) {
            if (!wait_row(s_col[ta])) { aborted = true; break; }
            waited = true;
            continue;
          }
        }
        waited = false;
        // pivots [ta, tb) are done: loads of their rows only after the flags (an acquire
        // at the IR level: nothing below is hoisted above the flag loads; no instruction)
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        for (int t = ta + lane; t < tb; t += 64) s_dk[t] = ld_sc1(rp, (unsigned)(s_kb[t] - kb0), VT());
        const int ua = s_off[ta], ub = s_off[tb];
        VT uv[UPL];
#pragma unroll
        for (int c = 0; c < UPL / PCH; c++)
          if (c * PCH * 64 < ub && (c + 1) * PCH * 64 > ua) {
#pragma unroll
            for (int m = c * PCH; m < (c + 1) * PCH; m++) uv[m] = ld_sc1(rp, offs[m], VT());
          }
#pragma unroll
        for (int c = 0; c < UPL / PCH; c++)
          if (c * PCH * 64 < ub && (c + 1) * PCH * 64 > ua) {
#pragma unroll
            for (int m = c * PCH; m < (c + 1) * PCH; m++) {
              const int u = lane + 64 * m;
              if (u >= ua && u < ub) {
                s_upos[u] = pp[m];
                s_uval[u] = uv[m];
              }
            }
          }
        wave_sync();
        // eliminate pivots [ta, tb); pivot t's diagonal position and value and this lane's
        // (at most two) entries of its row are read one pivot ahead
        auto load_piv = [&](int t, int& pik, VT& dk, int& pa, VT& ua_, int& pb, VT& ub_) {
          pik = s_pos[t];
          dk = s_dk[t];
          const int lo = s_off[t], hi = s_off[t + 1];
          const int e0 = lo + lane, e1 = e0 + 64;
          pa = 255; pb = 255; ua_ = (VT)0; ub_ = (VT)0;
          if (e0 < hi) { pa = s_upos[e0]; ua_ = s_uval[e0]; }
          if (e1 < hi) { pb = s_upos[e1]; ub_ = s_uval[e1]; }
        };
        int pik = 0, pa = 255, pb = 255;
        VT dk = (VT)1, va = (VT)0, vb = (VT)0;
        load_piv(ta, pik, dk, pa, va, pb, vb);
        for (int t = ta; t < tb; t++) {
          int pikn = 0, pan = 255, pbn = 255;
          VT dkn = (VT)1, van = (VT)0, vbn = (VT)0;
          if (t + 1 < tb) load_piv(t + 1, pikn, dkn, pan, van, pbn, vbn);
          const VT a = s_val[pik];
          const VT ca = pa != 255 ? s_val[pa] : (VT)0;
          const VT cb = pb != 255 ? s_val[pb] : (VT)0;
          const VT f = -a / dk;
          if (pa != 255) { const VT prod = f * va; s_val[pa] = ca + prod; }
          if (pb != 255) { const VT prod = f * vb; s_val[pb] = cb + prod; }
          wave_sync();
          if (lane == 0) s_val[pik] = f;           // the stored multiplier
          wave_sync();
          pik = pikn; dk = dkn; pa = pan; va = van; pb = pbn; vb = vbn;
        }
        ta = tb;
      }
    } else {
      for (int t0 = 0; t0 < nk && !aborted; t0 += 64) {
        const int t = t0 + lane;
        const bool ok = t >= nk || ld_flag(done + s_col[t]) == epoch;
        unsigned long long pending = __ballot(!ok);
        while (pending && !aborted) {
          if (!wait_row(s_col[t0 + (int)__builtin_ctzll(pending)])) aborted = true;
          pending &= pending - 1;
        }
      }
      if (!aborted) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        for (int t = lane; t < nk; t += 64) s_dk[t] = ld_sc1(rp, (unsigned)(s_kb[t] - kb0), VT());
        wave_sync();
        for (int t = 0; t < nk; t++) {
          const int k = s_col[t];
          const int pik = s_pos[t];
          const VT f = -s_val[pik] / s_dk[t];
          const int ua = s_off[t], ub = s_off[t + 1];
          for (int e = lane; e < ub - ua; e += 64) {
            const int q = s_kb[t] + 1 + e;
            const int cc = cols[q];
            int pos = 255;
            if (cc > k) {
              int lo = 0, hi = wi - 1;
              while (lo <= hi) {
                const int mid = (lo + hi) >> 1;
                const int v = s_col[mid];
                if (v == cc) { pos = s_pos[mid]; break; }
                if (v < cc) lo = mid + 1; else hi = mid - 1;
              }
            }
            if (pos != 255) {
              const VT prod = f * ld_sc1(rp, (unsigned)(q - kb0), VT());
              s_val[pos] = s_val[pos] + prod;
            }
          }
          wave_sync();
          if (lane == 0) s_val[pik] = f;
          wave_sync();
        }
      }
    }
    if (aborted) {
      if (lane == 0) st_flag(state + FLOW_ABORT, 1);
      break;
    }
    wave_sync();
    const __amdgpu_buffer_rsrc_t ro = sc1_rsrc(LU + p0);
    for (int t = lane; t < wi; t += 64) st_sc1(ro, (unsigned)t, s_val[t]);
    const bool bad = fabs((double)s_val[0]) < 1.0e-20;
    __builtin_amdgcn_s_waitcnt(0x0F70);            // vmcnt(0): the row is performed
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (lane == 0) {
      st_flag(done + i, epoch);
      if (bad) {
        atomicOr(state + FLOW_ERR, 1);
        atomicMin(state + FLOW_BADROW, i);
      }
    }
    wave_sync();                                   // LDS reused by the next row
  }
}

// ---- dataflow factorisation by units ----
//
// A unit is a node's rows (up to 3, one column set), and one wave factors it: lane l holds
// column l (and l + 64) of each row in registers, so that an entry of a pivot row is read once
// for all rows of the unit, a multiplier's way is two lane reads and one division (the rows'
// numerators side by side in its lanes), and the rows hand on to each other without leaving
// the wave.  What bounds the factorisation is the chain from a row to the next that needs it
// (store, flag, poll, load: some 3.4 us); the chain has a third of the links of the row-by-row
// kernel.  Pivot units are taken in ascending order as far as their flags are set; a finished
// unit's rows go out column by column (U: 3 words a column, from the unit's first row's own
// column on), and a plan (per pivot unit and lane: the column's place there, 255: none) makes
// the read of a pivot unit one load per lane.  Updates, order and rounding are those of
// k_ilu_flow.  FP32 at 200 x 20, 80 x 320, 640 x 320 cells: 1.25, 6.4, 17.5 ms, row by row 4.4,
// 19.5, 48; FP64 at 80 x 320 7.9 ms, row by row 21.8.

constexpr int FU = 3;             // rows of a unit
constexpr int FP = 64;            // pivot units of a unit

// desc: {first row, its CSR start, width | rows << 8 | pivot units << 16, own columns' place},
// {pivot list, plan (64-byte lines), place in U (columns), 0}; a pivot unit's entry: {place in
// U, place of its columns | its rows << 8, its last row, its position in desc}
struct FlowUnit { int r0, p0, w, rows, np, sd, list, line, ub; };
__device__ __forceinline__ FlowUnit flow_unit(const int4* __restrict__ desc, int k)
{
  const int4 a = desc[2 * k], b = desc[2 * k + 1];
  return { a.x, a.y, a.z & 255, (a.z >> 8) & 255, a.z >> 16, a.w, b.x, b.y, b.z };
}

__global__ void __launch_bounds__(64) k_unit_plan(const int4* __restrict__ desc,
                                                  const int4* __restrict__ list,
                                                  const int* __restrict__ srt_cols,
                                                  unsigned char* __restrict__ plan)
{
  const FlowUnit u = flow_unit(desc, blockIdx.x);
  const int slots = u.w > 64 ? 2 : 1;
  for (int t = 0; t < u.np; t++) {
    const FlowUnit v = flow_unit(desc, list[u.list + t].w);
    for (int c = 0; c < slots; c++) {
      const int l = threadIdx.x + 64 * c;
      int pos = 255;
      if (l < u.w) {
        const int cc = srt_cols[u.p0 + l];
        int lo = v.sd, hi = v.w - 1;
        while (lo <= hi) {
          const int mid = (lo + hi) >> 1;
          const int x = srt_cols[v.p0 + mid];
          if (x == cc) { pos = mid - v.sd; break; }
          if (x < cc) lo = mid + 1; else hi = mid - 1;
        }
      }
      plan[64LL * (u.line + t * slots + c) + threadIdx.x] = (unsigned char)pos;
    }
  }
}

__device__ __forceinline__ float lane_of(float x, int l)
{
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l));
}
__device__ __forceinline__ double lane_of(double x, int l)
{
  const u32x2 w = __builtin_bit_cast(u32x2, x);
  u32x2 r;
  r.x = (unsigned)__builtin_amdgcn_readlane((int)w.x, l);
  r.y = (unsigned)__builtin_amdgcn_readlane((int)w.y, l);
  return __builtin_bit_cast(double, r);
}
// column p of a row held in C registers a lane
template <class VT, int C>
__device__ __forceinline__ VT col_of(const VT* x, int p)
{
  if (C == 1) return lane_of(x[0], p);
  return p < 64 ? lane_of(x[0], p) : lane_of(x[C - 1], p - 64);
}

typedef unsigned u32x3 __attribute__((ext_vector_type(3)));
// the 3 words of column m (of a pivot unit's rows), sc1
__device__ __forceinline__ void ld_col(__amdgpu_buffer_rsrc_t r, unsigned m, float* v)
{
  const u32x3 w = __builtin_amdgcn_raw_buffer_load_b96(r, m * 12u, 0, 16);
  const unsigned x[3] = { w.x, w.y, w.z };
#pragma unroll
  for (int q = 0; q < 3; q++) v[q] = __builtin_bit_cast(float, x[q]);
}
__device__ __forceinline__ void ld_col(__amdgpu_buffer_rsrc_t r, unsigned m, double* v)
{
#pragma unroll
  for (int q = 0; q < 3; q++)
    v[q] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, m * 24u + 8u * q, 0, 16));
}
__device__ __forceinline__ void st_col(__amdgpu_buffer_rsrc_t r, unsigned m, float a, float b, float c)
{
  const u32x3 w = { __builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b),
                    __builtin_bit_cast(unsigned, c) };
  __builtin_amdgcn_raw_buffer_store_b96(w, r, m * 12u, 0, 16);
}
__device__ __forceinline__ void st_col(__amdgpu_buffer_rsrc_t r, unsigned m, double a, double b, double c)
{
  const double x[3] = { a, b, c };
#pragma unroll
  for (int q = 0; q < 3; q++)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x[q]), r, m * 24u + 8u * q, 0, 16);
}

// rows FROM.. of a unit minus their multiples of pivot row v (pivot dk, column place p): the
// rows' numerators go through one division
template <class VT, int C, int FROM>
__device__ __forceinline__ void unit_step(VT (&a)[FU][C], const VT* v, const bool* has, int p, VT dk)
{
#pragma clang fp contract(off)
  const int lane = threadIdx.x;
  VT num = col_of<VT, C>(a[FU - 1], p);
#pragma unroll
  for (int r = FU - 2; r >= FROM; r--) {
    const VT x = col_of<VT, C>(a[r], p);
    num = lane == r ? x : num;
  }
  const VT f = -num / dk;
#pragma unroll
  for (int r = FROM; r < FU; r++) {
    const VT fr = lane_of(f, r);
#pragma unroll
    for (int c = 0; c < C; c++) {
      const int l = lane + 64 * c;
      const VT prod = fr * v[c];
      const VT sum = a[r][c] + prod;
      a[r][c] = has[c] && l > p ? sum : a[r][c];
      a[r][c] = l == p ? fr : a[r][c];
    }
  }
}

// One unit; false: a wait was given up.
template <class VT, int C, class Wait>
__device__ __forceinline__ bool factor_unit(const FlowUnit& u, const int4* __restrict__ list,
                                            const unsigned char* __restrict__ plan,
                                            const unsigned char* __restrict__ srt_pos,
                                            VT* __restrict__ LU, VT* __restrict__ U, int* done,
                                            int epoch, int* state, unsigned char* s_plan,
                                            Wait wait_row)
{
  constexpr int B = sizeof(VT) == 4 ? 4 : 2;     // pivot units whose loads are in flight together
  const int lane = threadIdx.x;
  int pos[FU][C];
  VT a[FU][C];
#pragma unroll
  for (int r = 0; r < FU; r++)
#pragma unroll
    for (int c = 0; c < C; c++) {
      const int l = lane + 64 * c;
      pos[r][c] = r < u.rows && l < u.w ? (int)srt_pos[u.p0 + r * u.w + l] : 0;
    }
  int4 pv = {0, 0, 0, 0};
  if (lane < u.np) pv = list[u.list + lane];
  {
    const unsigned* src = reinterpret_cast<const unsigned*>(plan) + 16LL * u.line;
    unsigned* dst = reinterpret_cast<unsigned*>(s_plan);
    for (int k = lane; k < 16 * C * u.np; k += 64) dst[k] = src[k];
  }
#pragma unroll
  for (int r = 0; r < FU; r++)
#pragma unroll
    for (int c = 0; c < C; c++) {
      const int l = lane + 64 * c;
      a[r][c] = r < u.rows && l < u.w ? LU[u.p0 + r * u.w + pos[r][c]] : (VT)0;
    }
  wave_sync();
  int ta = 0;
  while (ta < u.np) {
    const bool ok = lane < ta || lane >= u.np || ld_flag(done + pv.z) == epoch;
    const unsigned long long pend = __ballot(!ok);
    int tb = pend ? (int)__builtin_ctzll(pend) : u.np;
    if (tb == ta) {                              // its flag was read last: it alone
      if (!wait_row(__builtin_amdgcn_readlane(pv.z, ta))) return false;
      tb = ta + 1;
    }
    // loads of the pivot units' rows only after their flags
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    for (int t0 = ta; t0 < tb; t0 += B) {
      VT v[B][C][FU];
      bool has[B][C];
#pragma unroll
      for (int b = 0; b < B; b++) {
        const int t = min(t0 + b, tb - 1);
        const __amdgpu_buffer_rsrc_t ru =
            sc1_rsrc(U + 3LL * __builtin_amdgcn_readlane(pv.x, t));
#pragma unroll
        for (int c = 0; c < C; c++) {
          const unsigned m = s_plan[64 * (t * C + c) + lane];
          has[b][c] = m != 255;
          ld_col(ru, m == 255 ? 0u : m, v[b][c]);
        }
      }
#pragma unroll
      for (int b = 0; b < B; b++)
        if (t0 + b < tb) {
          const int y = __builtin_amdgcn_readlane(pv.y, t0 + b);
          const int s0 = y & 255, rows = y >> 8;
#pragma unroll
          for (int q = 0; q < FU; q++)
            if (q < rows) {
              VT x[C];
#pragma unroll
              for (int c = 0; c < C; c++) x[c] = v[b][c][q];
              unit_step<VT, C, 0>(a, x, has[b], s0 + q, col_of<VT, C>(x, s0 + q));
            }
        }
    }
    ta = tb;
  }
  bool has[C];
#pragma unroll
  for (int c = 0; c < C; c++) has[c] = true;
  if (u.rows > 1) unit_step<VT, C, 1>(a, a[0], has, u.sd, col_of<VT, C>(a[0], u.sd));
  if (u.rows > 2) unit_step<VT, C, 2>(a, a[1], has, u.sd + 1, col_of<VT, C>(a[1], u.sd + 1));
  const __amdgpu_buffer_rsrc_t ro = sc1_rsrc(U + 3LL * u.ub);
#pragma unroll
  for (int c = 0; c < C; c++) {
    const int l = lane + 64 * c;
    if (l >= u.sd && l < u.w) st_col(ro, (unsigned)(l - u.sd), a[0][c], a[1][c], a[2][c]);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);            // vmcnt(0): the rows are performed
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  if (lane < u.rows) st_flag(done + u.r0 + lane, epoch);
#pragma unroll
  for (int r = 0; r < FU; r++)
    if (r < u.rows) {
#pragma unroll
      for (int c = 0; c < C; c++) {
        const int l = lane + 64 * c;
        if (l < u.w) LU[u.p0 + r * u.w + pos[r][c]] = a[r][c];
      }
      const VT d = col_of<VT, C>(a[r], u.sd + r);
      if (lane == 0 && fabs((double)d) < 1.0e-20) {
        atomicOr(state + FLOW_ERR, 1);
        atomicMin(state + FLOW_BADROW, u.r0 + r);
      }
    }
  return true;
}

template <class VT>
__global__ void __launch_bounds__(64) k_unit_flow(const int4* __restrict__ desc, int nu,
                                                  const int4* __restrict__ list,
                                                  const unsigned char* __restrict__ plan,
                                                  const unsigned char* __restrict__ srt_pos,
                                                  VT* __restrict__ LU, VT* __restrict__ U,
                                                  int* __restrict__ done, int epoch,
                                                  int* __restrict__ state, int spin_limit)
{
  __shared__ __attribute__((aligned(16))) unsigned char s_plan[FP * 128];
  const int lane = threadIdx.x;
  int polls = 0;
  auto wait_row = [&](int k) -> bool {
    for (;;) {
      int v = 0;
      if (lane == 0) v = ld_flag(done + k);
      if (__builtin_amdgcn_readfirstlane(v) == epoch) return true;
      if ((++polls & 31) == 0) {
        int ab = 0;
        if (lane == 0) ab = ld_flag(state + FLOW_ABORT);
        if (__builtin_amdgcn_readfirstlane(ab) != 0 || polls > spin_limit) return false;
      }
      __builtin_amdgcn_s_sleep(8);
    }
  };
  auto ticket = [&]() {
    int w = 0;
    if (lane == 0) w = __hip_atomic_fetch_add(state + FLOW_COUNTER, 1, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
    return __builtin_amdgcn_readfirstlane(w);
  };
  for (;;) {
    const int w = ticket();
    if (w >= nu) break;
    const FlowUnit u = flow_unit(desc, w);
    polls = 0;
    const bool ok = u.w > 64
        ? factor_unit<VT, 2>(u, list, plan, srt_pos, LU, U, done, epoch, state, s_plan, wait_row)
        : factor_unit<VT, 1>(u, list, plan, srt_pos, LU, U, done, epoch, state, s_plan, wait_row);
    if (!ok) {
      if (lane == 0) st_flag(state + FLOW_ABORT, 1);
      break;
    }
    wave_sync();                                   // LDS reused by the next unit
  }
}

// Pivot repair of row i (PRECO_ILU0::Factor, Preco_ilu0.cpp:95-135), every row before i
// final: among the rows eq > i of row i's pattern that hold column i, the one whose entry
// in column i is largest in magnitude (the first in row i's order on a tie) after its
// elimination by its pivot rows before i, is added to row i on row i's pattern.  The
// candidates' partial rows start from the matrix A (their factor rows may hold values of
// the failed pass).  One wave; state[FLOW_ERR] = 2 when no row qualifies.
__device__ __forceinline__ int row_pos(const int* __restrict__ srt_cols,
                                       const unsigned char* __restrict__ srt_pos, int q0, int w,
                                       int c)
{
  int lo = 0, hi = w - 1;
  while (lo <= hi) {
    const int mid = (lo + hi) >> 1;
    const int v = srt_cols[q0 + mid];
    if (v == c) return srt_pos[q0 + mid];
    if (v < c) lo = mid + 1; else hi = mid - 1;
  }
  return -1;
}

template <class VT>
__global__ void __launch_bounds__(64) k_ilu_repair(int i, const int* __restrict__ rp,
                                                   const int* __restrict__ cols,
                                                   const int* __restrict__ srt_cols,
                                                   const unsigned char* __restrict__ srt_pos,
                                                   const VT* __restrict__ A, VT* __restrict__ LU,
                                                   int* __restrict__ state)
{
#pragma clang fp contract(off)
  __shared__ VT s_v[FW], s_best[FW];
  const int lane = threadIdx.x;
  const int p0 = rp[i], wi = rp[i + 1] - p0;
  double bmax = 0.0;
  int best = -1, bq0 = 0, bw = 0;
  for (int j = 1; j < wi; j++) {
    const int eq = cols[p0 + j];
    if (eq <= i) continue;
    const int q0 = rp[eq], wq = rp[eq + 1] - q0;
    const int pos_i = row_pos(srt_cols, srt_pos, q0, wq, i);
    if (pos_i < 0) continue;
    for (int t = lane; t < wq; t += 64) s_v[t] = A[q0 + t];
    __syncthreads();
    // elimination by the pivot rows p < i of row eq, ascending
    for (int sidx = 0; sidx < wq; sidx++) {
      const int p = srt_cols[q0 + sidx];
      if (p >= i) break;
      const int pp = srt_pos[q0 + sidx];
      const int k0 = rp[p], wk = rp[p + 1] - k0;
      const VT f = -s_v[pp] / LU[k0];
      __syncthreads();
      for (int e = lane; e < wk - 1; e += 64) {
        const int q = k0 + 1 + e;
        const int c = cols[q];
        if (c > p) {
          const int pos = row_pos(srt_cols, srt_pos, q0, wq, c);
          if (pos >= 0) {
            const VT prod = f * LU[q];
            s_v[pos] = s_v[pos] + prod;
          }
        }
      }
      __syncthreads();
      if (lane == 0) s_v[pp] = f;
      __syncthreads();
    }
    const double m = fabs((double)s_v[pos_i]);
    if (m > bmax) {
      bmax = m;
      best = eq; bq0 = q0; bw = wq;
      for (int t = lane; t < wq; t += 64) s_best[t] = s_v[t];
    }
    __syncthreads();
  }
  if (best < 0) {
    if (lane == 0) state[FLOW_ERR] = 2;
    return;
  }
  for (int t = lane; t < wi; t += 64) {
    const int pos = row_pos(srt_cols, srt_pos, bq0, bw, cols[p0 + t]);
    if (pos >= 0) LU[p0 + t] = LU[p0 + t] + s_best[pos];
  }
}

// Completion flags of the rows after `from` cleared (their factorisation runs again).
__global__ void k_flags_clear(int from, int n, int* __restrict__ done)
{
  const int r = from + blockIdx.x * blockDim.x + threadIdx.x;
  if (r < n) done[r] = 0;
}

template <class VT>
__global__ void k_pack(long long ne, const int* __restrict__ psrc, const VT* __restrict__ LU,
                       VT* __restrict__ pval)
{
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < ne;
       t += (long long)gridDim.x * blockDim.x)
    pval[t] = psrc[t] >= 0 ? LU[psrc[t]] : (VT)0;       // negative: a zero (padding) entry
}

// Reciprocal diagonal in FP64 (1 for a negative source: an absent row).
template <class VT>
__global__ void k_pack_rcp(long long ne, const int* __restrict__ psrc, const VT* __restrict__ LU,
                           double* __restrict__ out)
{
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < ne;
       t += (long long)gridDim.x * blockDim.x)
    out[t] = psrc[t] >= 0 ? 1.0 / (double)LU[psrc[t]] : 1.0;
}

// Reciprocal diagonals in equation order.
template <class VT>
__global__ void k_rcp_diag(int n, const int* __restrict__ rowptr, const VT* __restrict__ LU,
                           double* __restrict__ out)
{
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r < n) out[r] = 1.0 / (double)LU[rowptr[r]];
}

template <class VT>
__global__ void k_pack_diag(int n, const int* __restrict__ prow, const int* __restrict__ rowptr,
                            const VT* __restrict__ LU, VT* __restrict__ pdiag)
{
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r < n) pdiag[r] = LU[rowptr[prow[r]]];
}

// ---------------------------------------------------------------------------------------
// sweeps

__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One lane's share of a row's sum over entries q0, q0 + G, ... below q1, each solved value
// from the LDS ring or, when it has left the ring, from the global copy (out of line: the
// sweeps take it only for long rows, wide levels and old dependencies).
template <class VT, int G>
__device__ __noinline__ double lane_sum(const VT* __restrict__ pval, const int* __restrict__ pcol,
                                        const double* ring, const double* __restrict__ xp,
                                        int q0, int q1, int lim)
{
  double s = 0.0;
  for (int q = q0; q < q1; q += G) {
    const int c = pcol[q];
    s += (double)pval[q] * (c >= lim ? ring[c & (RING - 1)] : xp[c]);
  }
  return s;
}

// Block b of the sweep: levels [blev[b], blev[b+1]) of the concatenated level table, rows
// at positions [bpos[b], bpos[b+1]).  Level offsets, columns and ring slots are local to
// the block; each block table has one extra sentinel level offset.
// The right-hand side of position r is gsrc[gidx[r]] (the input vector gathered into
// processing order on the fly); with oidx the solution of position r is also written to
// odst[oidx[r]] (scattered back to equation order).
// Sweep with a two-stage load pipeline and no global stores inside a level.  Level l
// computes from registers loaded during level l - 1 (stage 2: columns, values, right-hand
// side, diagonal); during level l the stage-2 loads of level l + 1 and the stage-1 loads
// of level l + 2 (row bounds, right-hand-side index) are issued, and every level starts by
// waiting for what the previous level issued, so no load is waited for in the level that
// issues it.  Results stay in the LDS ring and are flushed to the global copy (and the
// scatter target) at the full barriers: every FENCE positions, around wide levels and at
// the end.  A wide level (more than WIDE rows) reads and writes the global copy directly.
// With aidx, the scatter adds aval[aidx[e]] to the value written to odst[e] (the coarse
// prolongation P zc of the two-level preconditioner, folded into the write).
template <class VT, bool LOWER, int G, int PWN>
__global__ void __launch_bounds__(512) k_sweep_stage(const int* __restrict__ blev,
                                                     const int* __restrict__ bpos,
                                                     const int* __restrict__ lev_ptr_all,
                                                     const int* __restrict__ prs_all,
                                                     const int* __restrict__ pcol,
                                                     const VT* __restrict__ pval,
                                                     const VT* __restrict__ pdiag_all,
                                                     const int* __restrict__ gidx_all,
                                                     const double* __restrict__ gsrc,
                                                     const int* __restrict__ oidx_all,
                                                     double* __restrict__ odst,
                                                     double* __restrict__ xp_all,
                                                     const int* __restrict__ aidx,
                                                     const double* __restrict__ aval)
{
  __shared__ double ring[RING];
  __shared__ int s_lp[LPC + 2];
  const int b = blockIdx.x;
  const int lb = blev[b];
  const int nlev = blev[b + 1] - lb;
  const int* lev_ptr = lev_ptr_all + lb + 2 * b;   // nlev + 2 local offsets
  const int base = bpos[b];
  const int* prs = prs_all + base;
  const VT* pdiag = LOWER ? nullptr : pdiag_all + base;
  const int* gidx = gidx_all + base;
  const int* oidx = oidx_all ? oidx_all + base : nullptr;
  double* xp = xp_all + base;
  auto scatter = [&](int p, double v) {     // odst in equation order (+ the folded term)
    const int e = oidx[p];
    odst[e] = aidx ? v + aval[aidx[e]] : v;
  };
  const int t = threadIdx.x, nt = blockDim.x;
  const int grp = t / G, lane = t % G, ngr = nt / G;
  int lbase = 0;
  auto load_lp = [&](int l0) {
    for (int k = t; k < LPC + 2; k += nt) s_lp[k] = lev_ptr[min(l0 + k, nlev + 1)];
  };
  load_lp(0);
  __syncthreads();
  if (nlev <= 0) return;
  auto need_lp = [&](int L) {           // offsets of levels L and L + 1 staged
    if (L + 1 - lbase > LPC + 1) {
      __syncthreads();
      lbase = L - 1;
      load_lp(lbase);
      __syncthreads();
    }
  };
  int flushed = 0;                      // positions below are in the global copy
  // stage 1: row bounds and right-hand-side index of level [P_, P_ + nr_)
  auto stage1 = [&](int P_, int nr_, int& gi, int& qa, int& qb) {
    if (grp < nr_) {
      const int r = P_ + grp;
      gi = gidx[r];
      qa = prs[r];
      qb = prs[r + 1];
    }
  };
  // stage 2: right-hand side, diagonal, first PWN entries per lane
  auto stage2 = [&](int P_, int nr_, int gi, int qa, int qb, int* c, VT* v, double& in,
                    VT& dg) {
    if (grp < nr_) {
      in = gsrc[gi];
      if (!LOWER) dg = pdiag[P_ + grp];
#pragma unroll
      for (int j = 0; j < PWN; j++) {
        const int q = qa + lane + j * G;
        if (q < qb) { c[j] = pcol[q]; v[j] = pval[q]; }
        else { c[j] = -1; v[j] = (VT)0; }
      }
    }
  };
  int cN[PWN], cW[PWN];
  VT vN[PWN], vW[PWN];
  double inN = 0.0, inW = 0.0;
  VT dgN = (VT)1, dgW = (VT)1;
  int gi1 = 0, qa1 = 0, qb1 = 0, gi2 = 0, qa2 = 0, qb2 = 0, qaW = 0, qbW = 0;
#pragma unroll
  for (int j = 0; j < PWN; j++) { cN[j] = -1; vN[j] = (VT)0; cW[j] = -1; vW[j] = (VT)0; }
  // prologue: indices of levels 0 and 1, values of level 0
  int P0 = s_lp[0], nr0 = s_lp[1] - s_lp[0];
  int P1 = 0, nr1 = 0;
  stage1(P0, nr0, gi1, qa1, qb1);
  if (nlev > 1) {
    P1 = s_lp[1];
    nr1 = s_lp[2] - P1;
    stage1(P1, nr1, gi2, qa2, qb2);
  }
  stage2(P0, nr0, gi1, qa1, qb1, cN, vN, inN, dgN);
  for (int l = 0; l < nlev; l++) {
    // everything in flight was issued during the previous level
    __builtin_amdgcn_s_waitcnt(0x0F70);          // vmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < PWN; j++) { cW[j] = cN[j]; vW[j] = vN[j]; }
    inW = inN; dgW = dgN; qaW = qa1; qbW = qb1;
    gi1 = gi2; qa1 = qa2; qb1 = qb2;             // indices of level l + 1
    int P2 = 0, nr2 = 0;
    if (l + 2 < nlev) {
      need_lp(l + 2);
      P2 = s_lp[l + 2 - lbase];
      nr2 = s_lp[l + 3 - lbase] - P2;
    }
    __builtin_amdgcn_sched_barrier(0);
    if (l + 1 < nlev) stage2(P1, nr1, gi1, qa1, qb1, cN, vN, inN, dgN);
    if (l + 2 < nlev) stage1(P2, nr2, gi2, qa2, qb2);
    // level l: round 0 from the working registers, straight-line so that nothing issued
    // above is waited for; dependencies that left the ring, row tails beyond PWN entries
    // per lane and further rounds take the out-of-line path
    const int P = P0, nr = nr0;
    const bool wide = nr > WIDE;
    const int lim = wide ? INT_MAX : P + nr - RING;
    {
      const bool act = grp < nr;
      double s = 0.0;
      if (act) {
        bool old = false;
#pragma unroll
        for (int j = 0; j < PWN; j++) {
          const int cc = cW[j];
          if (cc >= 0) {
            old |= cc < lim;
            s += (double)vW[j] * ring[cc & (RING - 1)];
          }
        }
        if (old) {                           // dependencies that left the ring: global copy
          double xg[PWN];
#pragma unroll
          for (int j = 0; j < PWN; j++) {
            const int cc = cW[j];
            xg[j] = xp[(cc >= 0 && cc < lim) ? cc : 0];
          }
          s = 0.0;
#pragma unroll
          for (int j = 0; j < PWN; j++) {
            const int cc = cW[j];
            if (cc >= 0) {
              const double rv = ring[cc & (RING - 1)];
              s += (double)vW[j] * (cc < lim ? xg[j] : rv);
            }
          }
        }
        if (qbW > qaW + PWN * G)
          s += lane_sum<VT, G>(pval, pcol, ring, xp, qaW + lane + PWN * G, qbW, lim);
      }
#pragma unroll
      for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
      if (act && lane == 0) {
        const double xi = LOWER ? inW + s : (inW - s) / (double)dgW;
        ring[(P + grp) & (RING - 1)] = xi;
        if (wide) {
          xp[P + grp] = xi;
          if (oidx) scatter(P + grp, xi);
        }
      }
    }
    const int rounds = (nr + ngr - 1) / ngr;
    for (int k = 1; k < rounds; k++) {
      const int g = grp + k * ngr;
      const bool act = g < nr;
      double s = 0.0, in = 0.0;
      VT dg = (VT)1;
      if (act) {
        const int r = P + g;
        in = gsrc[gidx[r]];
        if (!LOWER) dg = pdiag[r];
        s = lane_sum<VT, G>(pval, pcol, ring, xp, prs[r] + lane, prs[r + 1], lim);
      }
#pragma unroll
      for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
      if (act && lane == 0) {
        const double xi = LOWER ? in + s : (in - s) / (double)dg;
        ring[(P + g) & (RING - 1)] = xi;
        if (wide) {
          xp[P + g] = xi;
          if (oidx) scatter(P + g, xi);
        }
      }
    }
    if (l + 1 >= nlev) break;
    const bool full = (P + nr) / FENCE != P / FENCE || wide || nr1 > WIDE;
    if (full) {
      if (!wide) {
        lds_barrier();
        for (int p = flushed + t; p < P + nr; p += nt) {
          const double v = ring[p & (RING - 1)];
          xp[p] = v;
          if (oidx) scatter(p, v);
        }
      }
      flushed = P + nr;
      __syncthreads();
    } else {
      lds_barrier();
    }
    P0 = P1; nr0 = nr1;
    P1 = P2; nr1 = nr2;
  }
  // the last level's results and whatever is still unflushed
  lds_barrier();
  if (nr0 <= WIDE)
    for (int p = flushed + t; p < P0 + nr0; p += nt) {
      const double v = ring[p & (RING - 1)];
      xp[p] = v;
      if (oidx) scatter(p, v);
    }
}

// ---------------------------------------------------------------------------------------
// block sweeps: one wave per block, both triangles in one launch

constexpr int BS_ROWS = 2047;      // rows per block
constexpr int BS_GROUP_ROWS = 4093; // rows per wave (12-bit positions)
constexpr int BS_WAVES = 1024;     // waves that fill the chip (one per SIMD)
constexpr int BS_SLOTS = 16;       // slots per pass (4 lanes each)
constexpr int BS_MAXW = 128;       // columns per node (8 slots of 16)
constexpr int BS_PAD = 64;         // padding after every stream (loads past the last node)
constexpr int BS_GATHER = 8;       // rows per lane whose loads are issued together
constexpr int BS_DEPTH = 4;        // passes whose loads are in flight ahead

// Slot descriptor: x = first row group of the slot's values (18 bits) | position of the
// node's first row << 18 (12 bits) | column groups in the slot - 1 << 30; y = first column
// group (16 bits) | node << 16 (12 bits) | rows << 28 (0: empty slot) | log2(slots of the
// node) << 30.  A node's slots are aligned to their number.  Descriptor 0 of a triangle is
// empty.
constexpr unsigned BS_VM = (1u << 18) - 1, BS_CM = (1u << 16) - 1, BS_PM = (1u << 12) - 1;

template <class VT> struct VQuad;
template <> struct VQuad<float> { using T = float4; using P = float2; };
template <> struct VQuad<double> { using T = double4; using P = double2; };

template <int C>
__device__ __forceinline__ double dpp_get(double v)
{
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), C, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), C, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
template <class T>
__device__ __forceinline__ T ld_off(const void* base, unsigned off)
{
  return *reinterpret_cast<const T*>(static_cast<const char*>(base) + off);
}
// doubles at a byte offset of the dynamic LDS (kernels without static LDS, as the set-up makes sure
// by lds_from_zero: it starts at 0, so the offset is the address; an address from the array's
// base takes one more instruction an access)
typedef __attribute__((address_space(3))) double lds_double;
__device__ __forceinline__ double ld_lds(unsigned off) { return *(const lds_double*)off; }
__device__ __forceinline__ void st_lds(unsigned off, double v) { *(lds_double*)off = v; }

// Row q's sum of a node in lane q of the node's first quad, from every lane's shares s0, s1,
// s2 of the three rows: two exchanges that halve the rows a lane carries, then, for nodes of
// more slots (lg: log2 of their number), the other quads' sums by row rotations and shuffles.
// M: the block has no such node, none of more than 2 slots, any.
template <int M>
__device__ __forceinline__ double node_sum(unsigned q, double s0, double s1, double s2, unsigned lg)
{
  const bool hi = q >= 2u, odd = q & 1u;
  double a = (hi ? s2 : s0) + dpp_get<0x4E>(hi ? s0 : s2);          // lane ^ 2
  double b = (hi ? 0.0 : s1) + dpp_get<0x4E>(hi ? s1 : 0.0);
  double s = (odd ? b : a) + dpp_get<0xB1>(odd ? a : b);            // lane ^ 1
  if (M > 0) {
    const double e = dpp_get<0x12C>(s);                             // the next quad's
    s += lg >= 1u ? e : 0.0;
    if (M > 1) {
      if (__any(lg > 1u)) {
        const double f = dpp_get<0x128>(s);                         // two quads on
        s += lg >= 2u ? f : 0.0;
        const double g = __shfl_xor(s, 16, 64);
        s += lg >= 3u ? g : 0.0;
      }
    }
  }
  return s;
}

// The node's rows solved across its first quad: row q in lane q from its right-hand side x
// and sum s.  Lower sweep (factors stored negated): x_q + s_q + l_q0 y_0 + l_q1 y_1, w the
// row's two couplings; upper sweep, last row first: (x_q - s_q - u_q2 y_2 - u_q1 y_1) rd, w =
// (u_q1, u_q2), rd the reciprocal diagonal.  Couplings a row does not have are zero.
template <bool LOWER, class W2>
__device__ __forceinline__ double node_solve(double x, double s, const W2& w, double rd)
{
  if (LOWER) {
    double t = x + s;
    t += (double)w.x * dpp_get<0x00>(t);
    t += (double)w.y * dpp_get<0x55>(t);
    return t;
  }
  double t = x - s;
  t -= (double)w.y * dpp_get<0xAA>(t * rd);
  t -= (double)w.x * dpp_get<0x55>(t * rd);
  return t * rd;
}

// The passes of one triangle of one block.  A pass holds up to 16 slots of 4 lanes; a slot
// holds up to 16 columns of one node, a node takes 1, 2, 4 or 8 neighbouring slots, and the
// nodes of a pass do not depend on each other.  Lane q of a slot multiplies column group q
// into the node's row sums; they end in the node's first slot, row r's in lane r (node_sum), the
// rows are solved across those lanes (node_solve) and lane r writes row r.  Column groups that a
// slot does not have read the block's zero group and the zero slot before x; rows that a node does
// not have read what follows and are not used.
// The chain from one pass to the next is one LDS read, four products, two exchanges (more for
// nodes of several slots), the node's solve and one LDS write, and a wave working alone is bound by its instructions
// (about 105 a pass, 4 cycles each; a branch costs about 70): nothing waits for memory, since
// values, columns, couplings and reciprocal diagonals are loaded D passes ahead into a
// register ring, the descriptors that name them 2 D, and the pass table's entries 3 D ahead.
// One wave works the block, so a pass ends without a workgroup barrier.
template <class VT, bool LOWER, int M, int D>
__device__ __forceinline__ void block_passes(int np, const unsigned* __restrict__ tab,
                                             const uint2* __restrict__ desc,
                                             const VT* __restrict__ vals,
                                             const uint2* __restrict__ cols,
                                             const VT* __restrict__ uval,
                                             const double* __restrict__ rdg, int lane)
{
  using V4 = typename VQuad<VT>::T;
  using V2 = typename VQuad<VT>::P;
  constexpr unsigned VB = sizeof(V4);
  const unsigned slot = lane >> 2, q = lane & 3;
  V4 va[D], vb[D], vc[D];
  V2 wu[D];
  double rd[D];
  uint2 ca[D], dr[D];
  unsigned xo[D], fl[D];                   // LDS offset of row q (0: none); the lane writes it,
                                           // log2 of the node's slots << 1
  // descriptors of D passes from the table's entries (one per lane)
  auto fetch = [&](unsigned t, uint2* d) {
#pragma unroll
    for (int k = 0; k < D; k++) {
      const unsigned s0 = __builtin_amdgcn_readlane(t, k), s1 = __builtin_amdgcn_readlane(t, k + 1);
      d[k] = desc[slot < s1 - s0 ? s0 + slot : 0u];
    }
  };
  const unsigned tl = min(lane, D);
  fetch(tab[tl], dr);
  tab += D;
  unsigned tv = tab[tl];
#pragma unroll
  for (int k = 0; k < D; k++) {             // the first D passes are empty
    ca[k] = make_uint2(0u, 0u);
    va[k] = vb[k] = vc[k] = V4{};
    wu[k] = V2{};
    rd[k] = 0.0;
    xo[k] = fl[k] = 0u;
    // waited for here: pending at the loop's entry, they would be waited for in every round,
    // with the loads in flight behind them
    asm volatile("" : "+v"(dr[k].x), "+v"(dr[k].y));
  }
  asm volatile("" : "+v"(tv));
  auto stage = [&](int k) {
    const uint2 d = dr[k];
    const unsigned R = d.y >> 28 & 3u, lg = d.y >> 30;
    const bool has = q <= d.x >> 30;
    ca[k] = ld_off<uint2>(cols, has ? ((d.y & BS_CM) + q) * 8u : 0u);
    const unsigned ov = has ? ((d.x & BS_VM) + q * R) * VB : 0u;
    va[k] = ld_off<V4>(vals, ov);
    vb[k] = ld_off<V4>(vals, ov + VB);
    vc[k] = ld_off<V4>(vals, ov + 2u * VB);
    const unsigned u = 4u * (d.y >> 16 & BS_PM) + q;
    wu[k] = ld_off<V2>(uval, u * (unsigned)sizeof(V2));
    if (!LOWER) rd[k] = ld_off<double>(rdg, u * 8u);
    xo[k] = q < R ? ((d.x >> 18 & BS_PM) + 1u + q) * 8u : 0u;
    fl[k] = (q < R && (M == 0 || (slot & ((1u << lg) - 1u)) == 0u) ? 1u : 0u) | lg << 1;
  };
  double h0 = 0.0;                          // right-hand side of the next pass's row
  auto pass = [&](int k) {
    const double xa = ld_lds(ca[k].x & 0xffffu), xc = ld_lds(ca[k].x >> 16);
    const double xd = ld_lds(ca[k].y & 0xffffu), xe = ld_lds(ca[k].y >> 16);
    // read a pass ahead (no other pass writes it), behind the reads that this pass waits for
    const double x0 = h0;
    h0 = ld_lds(xo[(k + 1) % D]);
    __builtin_amdgcn_sched_barrier(0);
    double s0 = (double)va[k].x * xa, s1 = (double)vb[k].x * xa, s2 = (double)vc[k].x * xa;
    s0 += (double)va[k].y * xc; s1 += (double)vb[k].y * xc; s2 += (double)vc[k].y * xc;
    s0 += (double)va[k].z * xd; s1 += (double)vb[k].z * xd; s2 += (double)vc[k].z * xd;
    s0 += (double)va[k].w * xe; s1 += (double)vb[k].w * xe; s2 += (double)vc[k].w * xe;
    const double s = node_sum<M>(q, s0, s1, s2, fl[k] >> 1);
    const double y = node_solve<LOWER>(x0, s, wu[k], rd[k]);
    // a wave's LDS operations complete in order: the compiler must keep the order, no wait
    asm volatile("" ::: "memory");
    if (fl[k] & 1u) st_lds(xo[k], y);
    asm volatile("" ::: "memory");
  };
  // no branch around a stage, so that every pass issues the same loads and the wait before
  // a pass's first use of its registers leaves the later passes' loads in flight; the first
  // D (empty) passes issue the loads of passes 0 .. D - 1, and the table's last entry is
  // repeated past the last pass (empty passes)
  for (int l0 = -D; l0 < np; l0 += D) {
    // the descriptors that the next D stages decode: asked for before anything else, so that
    // taking them over at the end leaves this round's loads in flight
    uint2 dn[D];
    fetch(tv, dn);
    tab += D;
    const unsigned tn = tab[tl];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < D; k++) {
      pass(k);
      stage(k);
    }
#pragma unroll
    for (int k = 0; k < D; k++) dr[k] = dn[k];
    tv = tn;
  }
}

// One block (or a group of independent blocks) per one-wave workgroup: its right-hand side is
// gathered into LDS (in local positions), swept down and up in place, and written back in equation order (with
// aidx, plus aval[aidx[e]]: the coarse prolongation folded into the write).  Blocks hold
// disjoint rows, so b and x may be the same vector.
template <class VT>
__global__ void __launch_bounds__(64) k_block_sweep(const int4* __restrict__ info,
                                                    const int* __restrict__ gidx,
                                                    const unsigned* __restrict__ tab,
                                                    const uint2* __restrict__ desc,
                                                    const VT* __restrict__ vlo,
                                                    const uint2* __restrict__ clo,
                                                    const VT* __restrict__ wlo,
                                                    const VT* __restrict__ vup,
                                                    const uint2* __restrict__ cup,
                                                    const VT* __restrict__ wup,
                                                    const double* __restrict__ rdg,
                                                    const double* rhs, double* out,
                                                    const int* __restrict__ aidx,
                                                    const double* __restrict__ aval)
{
  constexpr int G = BS_GATHER;
  extern __shared__ double smem[];
  const int4 i0 = info[4 * blockIdx.x], i1 = info[4 * blockIdx.x + 1];
  const int4 i2 = info[4 * blockIdx.x + 2], i3 = info[4 * blockIdx.x + 3];
  const int rb = i0.x, m = i0.y, ub = i0.z, tb = i0.w;
  const int lane = threadIdx.x;
  double* x = smem + 1;                                       // [m] local positions; [-1]: zero
  // gathers: every load of a chunk issued before any is waited for
  for (int k0 = 0; k0 < m; k0 += 64 * G) {
    int g[G];
    double v[G];
#pragma unroll
    for (int j = 0; j < G; j++) g[j] = gidx[rb + min(k0 + lane + 64 * j, m - 1)];
#pragma unroll
    for (int j = 0; j < G; j++) v[j] = rhs[g[j]];
#pragma unroll
    for (int j = 0; j < G; j++)
      if (k0 + lane + 64 * j < m) x[k0 + lane + 64 * j] = v[j];
  }
  if (lane < 3) smem[lane ? m + lane : 0] = 0.0;       // the zero slot, rows past the last
  wave_sync();
  auto lower = [&](auto mode) {
    block_passes<VT, true, decltype(mode)::value, BS_DEPTH>(
        i1.x, tab + tb, desc + i1.y, vlo + 4 * (long long)i2.x, clo + i2.y,
        wlo + 8 * (long long)ub, nullptr, lane);
  };
  auto upper = [&](auto mode) {
    block_passes<VT, false, decltype(mode)::value, BS_DEPTH>(
        i1.z, tab + tb + i1.x + 4 * BS_DEPTH, desc + i1.w, vup + 4 * (long long)i2.z, cup + i2.w,
        wup + 8 * (long long)ub, rdg + 4 * (long long)ub, lane);
  };
  if (i3.x == 0) lower(std::integral_constant<int, 0>());
  else if (i3.x == 1) lower(std::integral_constant<int, 1>());
  else lower(std::integral_constant<int, 2>());
  if (i3.y == 0) upper(std::integral_constant<int, 0>());
  else if (i3.y == 1) upper(std::integral_constant<int, 1>());
  else upper(std::integral_constant<int, 2>());
  wave_sync();
  for (int k0 = 0; k0 < m; k0 += 64 * G) {
    int e[G];
    double a[G];
#pragma unroll
    for (int j = 0; j < G; j++) e[j] = gidx[rb + min(k0 + lane + 64 * j, m - 1)];
    if (aidx) {
      int ai[G];
#pragma unroll
      for (int j = 0; j < G; j++) ai[j] = aidx[e[j]];
#pragma unroll
      for (int j = 0; j < G; j++) a[j] = aval[ai[j]];
    }
#pragma unroll
    for (int j = 0; j < G; j++) {
      const int k = k0 + lane + 64 * j;
      if (k < m) out[e[j]] = aidx ? x[k] + a[j] : x[k];
    }
  }
}

// ---------------------------------------------------------------------------------------
// node sweeps: one workgroup of several waves per block of any size

constexpr int NS_DEPTH = 4;        // passes whose loads are in flight ahead
constexpr int NS_WAVES = 4;        // waves per workgroup at most
constexpr int NS_LDS = 160 * 1024; // LDS of a workgroup at most (a double per live row)

// One triangle of one block by a workgroup of blockDim.x / 64 waves, as block_passes works
// it, with passes of up to blockDim.x / 4 slots (16 a wave) between LDS barriers.  A row's
// solved value lives in LDS from its pass to the last pass that reads it: the set-up gives
// every node LDS places as a linear scan allocates registers (place 0 holds the zero of
// absent columns), so a block may have far more rows than LDS holds values.  Right-hand
// sides are read and results written in equation order (a node's rows are consecutive
// equations); every row has its two couplings inside the node and its reciprocal diagonal.
// Descriptor: x = first row group of the slot's values | rows << 30 (0: empty); y = first
// column group | column groups in the slot - 1 << 30; z = the node's first equation | log2 of
// the node's slots << 30; w = its LDS place.  Group 0 of the streams is zero.
// What bounds it: one pass per level of nodes, about 1,100 cycles with four waves: the chain
// through LDS and a barrier, and every wave's loads through one CU's cache (64 bytes a cycle,
// empty slots included: eight waves take twice as long as four).  FP64, lower + upper sweep: a
// 200 x 20-cell channel (36,262 rows, 519 levels) 3.9 ms with the staged level sweeps, 0.51 ms
// here; a dried 80 x 320-cell meander (207,553 rows, 2,145 levels) 16.6 -> 3.2 ms.
template <class VT, bool LOWER, int M>
__global__ void __launch_bounds__(64 * NS_WAVES) k_node_sweep(const int4* __restrict__ info,
                                                              const unsigned* __restrict__ tabs,
                                                              const uint4* __restrict__ descs,
                                                              const VT* __restrict__ vals,
                                                              const uint2* __restrict__ cols,
                                                              const VT* __restrict__ wcp,
                                                              const double* __restrict__ rdg,
                                                              const double* rhs, double* out)
{
  using V4 = typename VQuad<VT>::T;
  using V2 = typename VQuad<VT>::P;
  constexpr unsigned IM = (1u << 30) - 1;
  constexpr int D = NS_DEPTH;
  extern __shared__ double smem[];
  const int4 in = info[blockIdx.x];                // passes, table, descriptors
  const int np = in.x;
  const unsigned* tab = tabs + in.y;
  const uint4* desc = descs + in.z;
  const int lane = threadIdx.x & 63;
  const unsigned slot = threadIdx.x >> 2, q = lane & 3;
  if (threadIdx.x == 0) smem[0] = 0.0;
  V4 va[D], vb[D], vc[D];
  V2 wu[D];
  double rd[D], hx[D];
  uint2 ca[D];
  uint4 dr[D];
  unsigned wo[D], fl[D], eo[D];            // LDS offset of the result (0: none), log2 of the
                                           // node's slots, equation of row q
  auto fetch = [&](unsigned t, uint4* d) {
#pragma unroll
    for (int k = 0; k < D; k++) {
      const unsigned s0 = __builtin_amdgcn_readlane(t, k), s1 = __builtin_amdgcn_readlane(t, k + 1);
      d[k] = desc[slot < s1 - s0 ? s0 + slot : 0u];
    }
  };
  const unsigned tl = min(lane, D);
  fetch(tab[tl], dr);
  tab += D;
  unsigned tv = tab[tl];
#pragma unroll
  for (int k = 0; k < D; k++) {             // the first D passes are empty
    ca[k] = make_uint2(0u, 0u);
    va[k] = vb[k] = vc[k] = V4{};
    wu[k] = V2{};
    rd[k] = hx[k] = 0.0;
    wo[k] = fl[k] = eo[k] = 0u;
    // waited for here (see block_passes)
    asm volatile("" : "+v"(dr[k].x), "+v"(dr[k].y), "+v"(dr[k].z), "+v"(dr[k].w));
  }
  asm volatile("" : "+v"(tv));
  auto stage = [&](int k) {
    const uint4 d = dr[k];
    const unsigned R = d.x >> 30, lg = d.z >> 30, e = d.z & IM;
    const bool has = q <= d.y >> 30;
    ca[k] = cols[has ? (d.y & IM) + q : 0u];
    const V4* v = reinterpret_cast<const V4*>(vals) + (has ? (d.x & IM) + q * R : 0u);
    va[k] = v[0];
    vb[k] = v[1];
    vc[k] = v[2];
    const unsigned eq = e + (q < R ? q : 0u);      // rows past the node's: its first again
    wu[k] = reinterpret_cast<const V2*>(wcp)[eq];
    if (!LOWER) rd[k] = rdg[eq];
    hx[k] = rhs[eq];
    wo[k] = q < R && (M == 0 || (slot & ((1u << lg) - 1u)) == 0u) ? (d.w + q) * 8u : 0u;
    eo[k] = eq;
    fl[k] = lg;
  };
  auto pass = [&](int k) {
    const double xa = ld_lds((ca[k].x & 0xffffu) * 8u), xc = ld_lds((ca[k].x >> 16) * 8u);
    const double xd = ld_lds((ca[k].y & 0xffffu) * 8u), xe = ld_lds((ca[k].y >> 16) * 8u);
    double s0 = (double)va[k].x * xa, s1 = (double)vb[k].x * xa, s2 = (double)vc[k].x * xa;
    s0 += (double)va[k].y * xc; s1 += (double)vb[k].y * xc; s2 += (double)vc[k].y * xc;
    s0 += (double)va[k].z * xd; s1 += (double)vb[k].z * xd; s2 += (double)vc[k].z * xd;
    s0 += (double)va[k].w * xe; s1 += (double)vb[k].w * xe; s2 += (double)vc[k].w * xe;
    const double s = node_sum<M>(q, s0, s1, s2, fl[k]);
    const double y = node_solve<LOWER>(hx[k], s, wu[k], rd[k]);
    if (wo[k]) {
      st_lds(wo[k], y);
      out[eo[k]] = y;
    }
    lds_barrier();
  };
  lds_barrier();
  for (int l0 = -D; l0 < np; l0 += D) {
    uint4 dn[D];
    fetch(tv, dn);
    tab += D;
    const unsigned tn = tab[tl];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < D; k++) {
      pass(k);
      stage(k);
    }
#pragma unroll
    for (int k = 0; k < D; k++) dr[k] = dn[k];
    tv = tn;
  }
}

// ---------------------------------------------------------------------------------------
// sweeps of blocks by chunks of 16 rows
//
// A block's triangular solve is a chain, of nodes if taken level by level (80 to 300 levels of
// some 700 cycles in a block of 700 rows), and what bounds it is the latency of a link, not its
// bytes.  A wave takes its block in the equations' own order, 16 rows at a time, with the
// inverse of the 16 x 16 triangle (k_chunk_inv, FP64, once per factorisation): a link is then
// the sparse sums over earlier chunks and one small product for 16 rows, 44 links a block.
// Lane 4 c + q works a quarter of row c's sum (columns as LDS byte offsets, two a packet and
// lane), then column c of the product for rows q, q + 4, q + 8, q + 12; the four are summed over
// the columns by two half-wave exchanges that also part the rows and two rotations, without a
// trip through LDS.  Packets and the inverse are loaded some chunks ahead, always the same number
// of loads (past a chunk's packets the next one's), so that the compiler's waits name the right
// ones.  Of the inverse the upper 4 x 4 blocks are not stored: plane j holds rows 4 j .. 4 j + 3,
// columns up to 4 j + 3.
// FP32, FP64 factors, both directions: 35, 33 us at 5,600 rows (60 x 13 quads), 35, 36 at 36,000,
// 39 at 231,000, 70, 84 at 923,000, 140, 164 at 1.8 million (3 TB/s); node by node 63, 43, 209, 251,
// 241 us (FP32).  A link takes 0.25 us (two packets a chunk) to 0.3 (four): some 280 cycles of
// dependent FP64 operations, an LDS write and read, the issue of the rest.  Matrix instructions for
// the row sums and the product are slower by a tenth (a dependent 4x4x4 FP64 one takes 50 cycles, an
// addition 28); chunks of 32 rows would take 1.6 times the bytes.
// A packet loaded past a chunk's own is the next chunk's; past a block's last chunk the stream
// holds packets of zeros that name the block's first row, so that LDS is read at the block's rows
// alone (what lies behind them is not written, and zero times a NaN is a NaN).

constexpr int CH_ROWS = 16;       // rows of a chunk
constexpr int CH_T = 160;         // stored entries of a chunk's inverse
// Up to this many blocks (3.5 waves a SIMD) the chain of a block is what counts; beyond, the
// bytes, of which the level sweep of several blocks a wave (k_block_sweep) takes half: 142 us
// against 219 at 3,072 blocks (1.8 million rows), 237 against 188 at 4,600, 607 against 353 at
// 12,300.
constexpr int CH_BLOCKS = 3584;
// Chunks in flight with two packets ahead each and with four (FP32, one less, this, and 6 and 4: 40,
// 39, 39 us at 231,000 rows with two packets; 37, 35, 34 at 36,000 and 43, 39, 37 at 145,000, cells
// of a channel, 139, 140, 139 at 1.8 million with four).
constexpr int CH_DEEP2 = 4, CH_DEEP = 3;
constexpr int CH_PK = 4;          // most packets of a chunk that are loaded ahead

__device__ __forceinline__ double2 swap32(double a, double b)
{
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a),
                                                   (unsigned)__double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a),
                                                   (unsigned)__double2hiint(b), false, false);
  const unsigned l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
  return make_double2(__hiloint2double((int)h0, (int)l0), __hiloint2double((int)h1, (int)l1));
}
__device__ __forceinline__ double2 swap16(double a, double b)
{
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a),
                                                   (unsigned)__double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a),
                                                   (unsigned)__double2hiint(b), false, false);
  const unsigned l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
  return make_double2(__hiloint2double((int)h0, (int)l0), __hiloint2double((int)h1, (int)l1));
}

template <class VT, int PK> struct ChunkBuf {
  VT v[PK][2];
  unsigned id[PK];
  double t[4], d;
  int pk;
};

// One direction: chunks in processing order (UP: from the block's end, rows of a chunk from its
// end).  cb: the block's first chunk, pb: its first packet; cnt: packets of every chunk.  A zero
// stands for what a row does not have (another chunk's packets, entries of the inverse), and zero
// times an infinity is a NaN: with ANY, the right-hand side may hold either, and such products are
// left out, so that they reach the rows that depend on them and no others.
template <class VT, int PK, bool UP, bool ANY>
__device__ __forceinline__ void chunk_sweep(int nch, int cb, int pb,
                                            const unsigned char* __restrict__ cnt,
                                            const unsigned* __restrict__ idx,
                                            const VT* __restrict__ val,
                                            const double* __restrict__ T,
                                            const double* __restrict__ D, unsigned spare)
{
  using P = typename VQuad<VT>::P;
  const int lane = threadIdx.x, c = lane >> 2, q = lane & 3;
  const unsigned cd = (lane < nch ? (unsigned)cnt[cb + lane] : 0u) |
                      (64 + lane < nch ? (unsigned)cnt[cb + 64 + lane] : 0u) << 16;
  auto packets = [&](int t) {
    const unsigned long long d = (unsigned)__builtin_amdgcn_readlane((int)cd, t & 63);
    return (int)(d >> ((t >> 6) * 16) & 0xFFFF);
  };
  const int t0 = min(lane, 15), t1 = 16 + min(lane, 31), t2 = 48 + min(lane, 47), t3 = 96 + lane;
  const unsigned* ip = idx + (size_t)pb * 64;
  const P* vp = reinterpret_cast<const P*>(val) + (size_t)pb * 64;
  const double* tp = T + (size_t)cb * CH_T;
  const double* dp = UP ? D + (size_t)cb * CH_ROWS + c : nullptr;
  int pk = 0;
  auto load = [&](ChunkBuf<VT, PK>& b, int t) {
#pragma unroll
    for (int p = 0; p < PK; p++) {
      b.id[p] = ip[64 * p + lane];
      const P w = vp[64 * p + lane];
      b.v[p][0] = w.x; b.v[p][1] = w.y;
    }
    b.t[0] = tp[t0]; b.t[1] = tp[t1]; b.t[2] = tp[t2]; b.t[3] = tp[t3];
    if (UP) { b.d = *dp; dp += CH_ROWS; }
    b.pk = pk;
    const int np = packets(t);
    ip += 64 * np;
    vp += 64 * np;
    tp += CH_T;
    pk += np;
  };
  const bool keep = (c & 3) == q;                  // the lane's own row is its row of the product
  const int r = 4 * (lane >> 4) + q;
  unsigned own = 8u * (UP ? CH_ROWS * nch - 1 - c : c), to = 8u * (UP ? CH_ROWS * nch - 1 - r : r);
  // a chunk's reads of LDS; its packets 2 and 3 (the last of 2 or 4 may be another chunk's) are
  // read where it has more than 2
  double x[2 * PK], s0;
  int np;
  auto fetch = [&](const ChunkBuf<VT, PK>& b, int t) {
    np = packets(t);
#pragma unroll
    for (int p = 0; p < 2; p++) {
      x[2 * p] = ld_lds(b.id[p] & 0xFFFFu);
      x[2 * p + 1] = ld_lds(b.id[p] >> 16);
    }
    if (PK > 2 && np > 2) {
#pragma unroll
      for (int p = 2; p < PK; p++) {
        x[2 * p] = ld_lds(b.id[p] & 0xFFFFu);
        x[2 * p + 1] = ld_lds(b.id[p] >> 16);
      }
    }
    s0 = ld_lds(own);
    own += UP ? -8u * CH_ROWS : 8u * CH_ROWS;
  };
  auto step = [&](const ChunkBuf<VT, PK>& b) {
    auto f = [](VT v) { return UP ? -(double)v : (double)v; };
    if (ANY) {
#pragma unroll
      for (int p = 1; p < PK; p++)
        if (p >= np) x[2 * p] = x[2 * p + 1] = 0.0;
    }
    double a0 = f(b.v[0][0]) * x[0], a1 = f(b.v[0][1]) * x[1];
    a0 += f(np > 1 ? b.v[1][0] : (VT)0) * x[2];
    a1 += f(np > 1 ? b.v[1][1] : (VT)0) * x[3];
    if (np > 2) {
      if (PK > 2) {
#pragma unroll
        for (int p = 2; p < PK; p++) {
          a0 += f(p < PK - 1 || np > p ? b.v[p][0] : (VT)0) * x[2 * p];
          a1 += f(p < PK - 1 || np > p ? b.v[p][1] : (VT)0) * x[2 * p + 1];
        }
      }
      for (int p = PK; p < np; p++) {
        const size_t at = (size_t)(pb + b.pk + p) * 64 + lane;
        const unsigned id = idx[at];
        const P w = reinterpret_cast<const P*>(val)[at];
        a0 += f(w.x) * ld_lds(id & 0xFFFFu);
        a1 += f(w.y) * ld_lds(id >> 16);
      }
    }
    a0 += a1;
    a0 += dpp_get<0xB1>(a0);                       // over the row's four lanes
    a0 += dpp_get<0x4E>(a0);
    const double s = s0 + a0;
    auto times = [&](double t) { return ANY && t == 0.0 ? 0.0 : t * s; };
    const double p0 = times(lane < 16 ? b.t[0] : 0.0), p1 = times(lane < 32 ? b.t[1] : 0.0);
    const double p2 = times(lane < 48 ? b.t[2] : 0.0), p3 = times(b.t[3]);
    const double2 e = swap32(p0, p2), h = swap32(p1, p3);
    const double2 g = swap16(e.x + e.y, h.x + h.y);
    double y = g.x + g.y;
    y += dpp_get<0x128>(y);                        // 8 lanes on
    const double own_part = UP ? b.d * s + y : s + y;
    st_lds(keep ? to : spare, own_part + dpp_get<0x124>(y));
    to += UP ? -8u * CH_ROWS : 8u * CH_ROWS;
  };
  constexpr int R = PK == 2 ? CH_DEEP2 : CH_DEEP;
  ChunkBuf<VT, PK> buf[R];
#pragma unroll
  for (int u = 0; u < R; u++) load(buf[u], u);
  fetch(buf[0], 0);
  for (int t = 0;; t += R) {
#pragma unroll
    for (int u = 0; u < R; u++) {
      step(buf[u]);
      if (t + u + 1 >= nch) return;
      fetch(buf[(u + 1) % R], t + u + 1);
      asm volatile("" ::: "memory");               // the loads ahead while LDS answers
      load(buf[u], t + u + R);
    }
  }
}

template <class VT, int PK>
__global__ void __launch_bounds__(64) k_chunk_sweep(const int4* __restrict__ info,
                                                    const int* __restrict__ rows,
                                                    const unsigned char* __restrict__ dlo,
                                                    const unsigned* __restrict__ ilo,
                                                    const VT* __restrict__ vlo,
                                                    const double* __restrict__ tlo,
                                                    const unsigned char* __restrict__ dup,
                                                    const unsigned* __restrict__ iup,
                                                    const VT* __restrict__ vup,
                                                    const double* __restrict__ tup,
                                                    const double* __restrict__ dgu,
                                                    const double* __restrict__ b,
                                                    double* __restrict__ x,
                                                    const int* __restrict__ aidx,
                                                    const double* __restrict__ aval)
{
  constexpr int U = 16;                            // rows a lane in flight
  const int lane = threadIdx.x;
  const int4 w0 = info[2 * blockIdx.x], w1 = info[2 * blockIdx.x + 1];
  const int m = w0.y, nch = (m + CH_ROWS - 1) / CH_ROWS, all = nch * CH_ROWS;
  const int* row = rows + w0.x;
  bool finite = true;
  for (int k0 = 0; k0 < all; k0 += 64 * U) {
    int i[U];
    double v[U];
#pragma unroll
    for (int u = 0; u < U; u++) i[u] = row[min(k0 + 64 * u + lane, m - 1)];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = b[i[u]];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = k0 + 64 * u + lane;
      finite = finite && __builtin_isfinite(v[u]);
      if (k < all) st_lds(8u * k, k < m ? v[u] : 0.0);
    }
  }
  asm volatile("" ::: "memory");
  const unsigned spare = 8u * (all + lane);
  if (__all(finite)) {
    chunk_sweep<VT, PK, false, false>(nch, w0.z, w1.x, dlo, ilo, vlo, tlo, nullptr, spare);
    asm volatile("" ::: "memory");
    chunk_sweep<VT, PK, true, false>(nch, w0.z, w1.y, dup, iup, vup, tup, dgu, spare);
  } else {
    chunk_sweep<VT, PK, false, true>(nch, w0.z, w1.x, dlo, ilo, vlo, tlo, nullptr, spare);
    asm volatile("" ::: "memory");
    chunk_sweep<VT, PK, true, true>(nch, w0.z, w1.y, dup, iup, vup, tup, dgu, spare);
  }
  asm volatile("" ::: "memory");
  for (int k0 = 0; k0 < m; k0 += 64 * U) {
    int i[U];
    double v[U];
#pragma unroll
    for (int u = 0; u < U; u++) i[u] = row[min(k0 + 64 * u + lane, m - 1)];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = aidx ? aval[aidx[i[u]]] : 0.0;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = k0 + 64 * u + lane;
      if (k < m) x[i[u]] = ld_lds(8u * k) + v[u];
    }
  }
}

// Inverses of a chunk's triangles, one wave a chunk.  Both are taken as lower ones in processing
// order: row r is (e_r + sum of g_rk times row k) / d_r, with g the stored (negated) multipliers
// and d = 1 below, g = -u and d = u_rr above.  In twice FP64's digits (error-free sums and
// products), so that the product with the inverse has only the rounding of its entries on top of
// its own, and with the diagonals kept apart: a row's own term is added last.  The error of an
// apply against extended precision is then that of a substitution (18 meshes: 1.0 times that of
// the level sweeps where both are near rounding, 0.6 to 5 times, 1.3 in the mean, where the
// factors amplify it; two orders of the same substitution differ as much).
template <class VT>
__global__ void __launch_bounds__(64) k_chunk_inv(const int4* __restrict__ chunks,
                                                  const int* __restrict__ rows,
                                                  const int* __restrict__ slot,
                                                  const int* __restrict__ rp,
                                                  const int* __restrict__ cols,
                                                  const VT* __restrict__ LU,
                                                  double* __restrict__ tlo, double* __restrict__ tup,
                                                  double* __restrict__ dgu)
{
#pragma clang fp contract(off)
  __shared__ double G[2][CH_ROWS][CH_ROWS + 1], D[2][CH_ROWS];
  const int lane = threadIdx.x, h = blockIdx.x;
  const int4 ch = chunks[h];                       // first row, rows, place in tlo, in tup
  for (int k = lane; k < 2 * CH_ROWS * (CH_ROWS + 1); k += 64) (&G[0][0][0])[k] = 0.0;
  if (lane < 2 * CH_ROWS) (&D[0][0])[lane] = 1.0;
  __syncthreads();
  const int r = lane >> 2, q = lane & 3;
  if (r < ch.y) {
    const int i = rows[ch.x + r], p0 = rp[i], p1 = rp[i + 1];
    if (q == 0) D[1][CH_ROWS - 1 - r] = (double)LU[p0];
    for (int e = p0 + 1 + q; e < p1; e += 4) {
      const int j = cols[e], sl = slot[j];
      if ((sl >> 4) != h) continue;
      const int k = sl & (CH_ROWS - 1);
      if (k < r) G[0][r][k] = (double)LU[e];
      else G[1][CH_ROWS - 1 - r][CH_ROWS - 1 - k] = -(double)LU[e];
    }
  }
  __syncthreads();
  if (lane >= 2 * CH_ROWS) return;
  const int dir = lane >> 4, c = lane & 15;
  double* T = dir ? tup + (size_t)ch.w * CH_T : tlo + (size_t)ch.z * CH_T;
  double z[CH_ROWS], zl[CH_ROWS];
#pragma unroll
  for (int k = 0; k < CH_ROWS; k++) {
    double s = k == c ? 1.0 : 0.0, sl = 0.0;
#pragma unroll
    for (int l = 0; l < k; l++) {
      const double g = G[dir][k][l], p = g * z[l], e = fma(g, z[l], -p);
      const double t = s + p, v = t - s;
      sl += fma(g, zl[l], e) + ((s - (t - v)) + (p - v));
      s = t;
    }
    const double d = D[dir][k], q = s / d, r = (fma(-q, d, s) + sl) / d;
    z[k] = q + r;
    zl[k] = r - (z[k] - q);
    const int j = k >> 2;
    if (c < 4 * (j + 1)) T[8 * j * (j + 1) + 4 * c + (k & 3)] = k == c ? 0.0 : z[k];
    if (dir && k == c) dgu[(size_t)ch.w * CH_ROWS + c] = z[k];
  }
}

// ---------------------------------------------------------------------------------------
// host set-up

// RMX_SWEEP selects the sweep kernels (tuning and comparison), read when a system is set up
// and at every application: 1 the staged level sweeps; 2 the block sweeps where every block has
// at most BS_ROWS rows, else the node sweeps where the rows alive at a time fit LDS, else 1;
// 3 (default) the chunk sweeps of the strip ILU(0) where its blocks fit them, else 2.
static int sweep_variant()
{
  const char* e = getenv("RMX_SWEEP");
  return e ? atoi(e) : 3;
}

// Fails where one of the kernels that take LDS offsets for addresses has LDS of its own.
template <class... K>
static void lds_from_zero(K*... kernels)
{
  for (const void* k : { (const void*)kernels... }) {
    hipFuncAttributes a;
    HIPCHECK(hipFuncGetAttributes(&a, k));
    if (a.sharedSizeBytes != 0) fail(RMX_ERR_HIP, "sweeps: dynamic LDS does not start at address 0");
  }
}

// Level sets of the lower or upper dependency graph of rows [a, e), entries with a column
// outside [a, e) or (with `seg`) in another segment ignored.
static void levels(int a, int e, const std::vector<int>& rp, const std::vector<int>& cl, bool lower,
                   const std::vector<int>& seg, std::vector<int>& lev, std::vector<int>& ptr,
                   std::vector<int>& rows)
{
  int nlev = 0;
  const bool sg = !seg.empty();
  if (lower) {
    for (int i = a; i < e; i++) {
      int l = 0;
      for (int q = rp[i] + 1; q < rp[i + 1]; q++)
        if (cl[q] < i && cl[q] >= a && (!sg || seg[cl[q]] == seg[i])) l = std::max(l, lev[cl[q]] + 1);
      lev[i] = l;
      nlev = std::max(nlev, l + 1);
    }
  } else {
    for (int i = e - 1; i >= a; i--) {
      int l = 0;
      for (int q = rp[i] + 1; q < rp[i + 1]; q++)
        if (cl[q] > i && cl[q] < e && (!sg || seg[cl[q]] == seg[i])) l = std::max(l, lev[cl[q]] + 1);
      lev[i] = l;
      nlev = std::max(nlev, l + 1);
    }
  }
  ptr.assign(nlev + 1, 0);
  for (int i = a; i < e; i++) ptr[lev[i] + 1]++;
  for (int l = 0; l < nlev; l++) ptr[l + 1] += ptr[l];
  rows.assign(e - a, 0);
  std::vector<int> fill(ptr.begin(), ptr.end() - 1);
  if (lower) { for (int i = a; i < e; i++) rows[fill[lev[i]]++] = i; }
  else { for (int i = e - 1; i >= a; i--) rows[fill[lev[i]]++] = i; }
}

// Rows of the levels of every strip, levels of more than cap rows split: per strip its first
// level and position, per level its first position (and one more, a sentinel).
static void strip_levels(SweepSet& S, const Ilu& I, bool lower, int cap, std::vector<int>& blev,
                         std::vector<int>& bpos, std::vector<int>& levp, std::vector<int>& prow)
{
  const int n = I.n, nb = I.nblk;
  const std::vector<int>& rp = I.h_rp;
  const std::vector<int>& cl = I.h_cols;
  std::vector<int> lev(n, 0);
  blev.assign(nb + 1, 0); bpos.assign(nb + 1, 0); levp.clear(); prow.clear();
  levp.reserve(n / 8);
  prow.reserve(n);
  int maxnr = 0, nlev_tot = 0;
  for (int b = 0; b < nb; b++) {
    const int a = I.bstart[b], e = I.bstart[b + 1];
    std::vector<int> ptr, rows;
    levels(a, e, rp, cl, lower, I.seg, lev, ptr, rows);
    if (cap > 0) {                                 // levels of more than cap rows split
      std::vector<int> cp(1, 0);
      for (size_t l = 0; l + 1 < ptr.size(); l++)
        for (int r = ptr[l]; r < ptr[l + 1]; r += cap) cp.push_back(std::min(r + cap, ptr[l + 1]));
      ptr.swap(cp);
    }
    const int nl = (int)ptr.size() - 1;
    blev[b + 1] = blev[b] + nl;
    bpos[b + 1] = bpos[b] + (e - a);
    for (int l = 0; l <= nl; l++) levp.push_back(ptr[l]);
    levp.push_back(ptr[nl]);                       // sentinel: lev_ptr[l+2] for the last level
    for (int l = 0; l < nl; l++) maxnr = std::max(maxnr, ptr[l + 1] - ptr[l]);
    prow.insert(prow.end(), rows.begin(), rows.end());
    nlev_tot = std::max(nlev_tot, nl);
  }
  S.nlev_max = nlev_tot;
  S.max_nr = maxnr;
  S.nlev_sum = blev[nb];
}

// Entries that the sweeps of I keep: the strict lower / upper part inside a row's strip and segment.
static void count_entries(Ilu& I)
{
  std::atomic<long long> lo{0}, up{0};
  const bool sg = !I.seg.empty();
  std::vector<int> blk(I.nblk > 1 ? I.n : 0);
  if (I.nblk > 1)
    for (int b = 0; b < I.nblk; b++) std::fill(blk.begin() + I.bstart[b], blk.begin() + I.bstart[b + 1], b);
  parallel_for(I.n, [&](long long a, long long e) {
    long long l = 0, u = 0;
    for (long long i = a; i < e; i++)
      for (int q = I.h_rp[i] + 1; q < I.h_rp[i + 1]; q++) {
        const int c = I.h_cols[q];
        if ((I.nblk > 1 && blk[c] != blk[i]) || (sg && I.seg[c] != I.seg[i])) continue;
        l += c < i;
        u += c > i;
      }
    lo += l;
    up += u;
  });
  I.lo.ne = lo;
  I.up.ne = up;
}

// Levels of a system whose sweeps do not walk them, worked out where they are asked for.
void sweep_levels(Ilu& I)
{
  std::vector<int> blev, bpos, levp, prow;
  if (I.lo.nlev_max < 0) strip_levels(I.lo, I, true, I.level_cap, blev, bpos, levp, prow);
  if (I.up.nlev_max < 0) strip_levels(I.up, I, false, I.level_cap, blev, bpos, levp, prow);
}

// Packed layout of one sweep over all blocks.
static void build_sweep(SweepSet& S, const Ilu& I, bool lower, std::vector<int>& order, hipStream_t s)
{
  const int n = I.n, nb = I.nblk;
  const std::vector<int>& rp = I.h_rp;
  const std::vector<int>& cl = I.h_cols;
  std::vector<int> blev, bpos, levp, prow;
  strip_levels(S, I, lower, I.level_cap, blev, bpos, levp, prow);
  // positions: local to each block
  std::vector<int> pos(n);
  for (int b = 0; b < nb; b++)
    for (int r = bpos[b]; r < bpos[b + 1]; r++) pos[prow[r]] = r - bpos[b];
  // entries of row i kept by the sweep: the strict lower / upper part inside i's strip
  std::vector<int> blk(n);
  for (int b = 0; b < nb; b++)
    for (int i = I.bstart[b]; i < I.bstart[b + 1]; i++) blk[i] = b;
  const bool sg = !I.seg.empty();
  auto keep = [&](int i, int c) {
    return (lower ? c < i : c > i) && c >= I.bstart[blk[i]] && c < I.bstart[blk[i] + 1] &&
           (!sg || I.seg[c] == I.seg[i]);
  };
  std::vector<int> prs(n + 1, 0);
  parallel_for(n, [&](long long a, long long b) {
    for (long long r = a; r < b; r++) {
      const int i = prow[r];
      int k = 0;
      for (int q = rp[i] + 1; q < rp[i + 1]; q++) k += keep(i, cl[q]);
      prs[r + 1] = k;
    }
  });
  for (int r = 0; r < n; r++) prs[r + 1] += prs[r];
  const long long ne = prs[n];
  std::vector<int> pcol(ne), psrc(ne);
  parallel_for(n, [&](long long a, long long b) {
    for (long long r = a; r < b; r++) {
      const int i = prow[r];
      int j = prs[r];
      for (int q = rp[i] + 1; q < rp[i + 1]; q++)
        if (keep(i, cl[q])) { pcol[j] = pos[cl[q]]; psrc[j] = q; j++; }
    }
  });
  S.nblk = nb;
  S.ne = ne;
  if (getenv("RMX_DEBUG"))
    fprintf(stderr, "[rmx] %s sweep, %d strip(s) x %d segment(s): %d levels (longest strip), "
            "%.1f rows/level, max %d, %lld entries\n", lower ? "lower" : "upper", nb, I.nseg,
            S.nlev_max, (double)n / std::max(1, S.nlev_sum), S.max_nr, ne);
  S.packed = true;
  S.blev.upload(blev, s); S.bpos.upload(bpos, s); S.lev_ptr.upload(levp, s);
  S.prs.upload(prs, s); S.prow.upload(prow, s); S.pcol.upload(pcol, s); S.psrc.upload(psrc, s);
  HIPCHECK(hipStreamSynchronize(s));
  order = prow;
}

// Block sweep layout.  A block is the rows of one strip in one segment, and a wave works a
// group of blocks of one strip (below, the layout of a group); a unit is a run of
// rows of one node (group), at most 3 (every row its own unit without `group`).  Unit
// levels: a unit's lower level is one more than the highest of the units its rows couple to
// below them in the block (upper: above); units of a level are independent.  A unit's
// columns are the union of its rows' columns outside the unit (the rows of a node have the
// same ones), in groups of 4 (zero-padded), a slot for every 4 groups, the slots rounded up
// to a power of two (the added ones hold no columns).  Units of a level are listed by
// falling slot count, so that a unit's slots are aligned to their number, and cut into
// passes of at most 16 slots.  Local positions list the units in lower order, a unit's rows
// together.  The first column group and the first 3 row groups of a block's streams are zero.
// Entries keep the strip sweeps' rule (the strict triangle inside the row's
// block), minus the couplings inside a unit, which go to the unit's record.  Off (the node
// sweeps run) when a block has more than BS_ROWS rows or a group does not fit the
// descriptors.
// scol, spos: every row's columns ascending and their places in the row.
static void build_blocks(Ilu& I, const std::vector<int>* group, const std::vector<int>& scol,
                         const std::vector<unsigned char>& spos, hipStream_t s)
{
  BlockSweep& B = I.bs;
  B.on = false;
  const int n = I.n, nstrip = I.nblk, nseg = std::max(1, I.nseg);
  const std::vector<int>& rp = I.h_rp;
  const bool sg = !I.seg.empty();
  auto segof = [&](int i) { return sg ? I.seg[i] : 0; };
  if (nseg == 1)
    for (int b = 0; b < nstrip; b++)
      if (I.bstart[b + 1] - I.bstart[b] > BS_ROWS) return;
  // tighter pass caps (tests of the level split): rows and entry pairs (each row's entries in
  // pairs, at least one) of a pass; a node needing more sits alone
  int cap_rows = 3 * BS_SLOTS, cap_pairs = INT_MAX;
  if (const char* e = getenv("RMX_BLOCK_LEVEL_ROWS")) cap_rows = std::max(3, std::min(cap_rows, atoi(e)));
  if (const char* e = getenv("RMX_BLOCK_LEVEL_PAIRS")) cap_pairs = std::max(1, atoi(e));
  // CSR position of entry (r, c), -1 if the pattern has none
  auto find = [&](int r, int c) {
    const auto b = scol.begin() + rp[r], e = scol.begin() + rp[r + 1];
    const auto it = std::lower_bound(b, e, c);
    return it != e && *it == c ? rp[r] + (int)spos[it - scol.begin()] : -1;
  };
  struct Part {
    std::vector<int> rows;               // equation at every local position
    std::vector<unsigned> tab[2];        // pass tables: first slot of every pass (lower, upper)
    std::vector<uint2> desc[2];          // slot descriptors
    int npass[2] = {0, 0}, lgmax[2] = {0, 0};   // lgmax: log2 of the most slots of a node
    std::vector<unsigned short> col[2];  // columns, LDS byte offsets, 4 per group
    std::vector<int> src[2];             // CSR position of every value (4 per row group)
    std::vector<int> usrc[2];            // unit coupling sources (2 per row, 4 rows per unit)
    std::vector<int> dsrc;               // unit diagonal sources (4 per unit)
    bool fits = true;
  };
  // Blocks per wave: neighbouring segments of a strip share a wave, level by level, where a
  // wave per block would leave each SIMD more than one (their levels hold a few nodes each,
  // so a wave alone uses a few of its 16 slots and the chip issues mostly empty lanes): about
  // BS_WAVES groups in all (RMX_BLOCK_WAVES: fewer or more, for tests of their size), of at most
  // BS_GROUP_ROWS rows.
  int waves = BS_WAVES;
  if (const char* e = getenv("RMX_BLOCK_WAVES")) waves = std::max(1, atoi(e));
  std::vector<int> gps(nstrip, nseg);          // groups of every strip
  for (int b = 0; b < nstrip; b++) {
    const int rows = I.bstart[b + 1] - I.bstart[b];
    int k = std::max(1, std::min(nseg, (waves + nstrip - 1) / nstrip));
    while (k < nseg && (long long)rows * ((nseg + k - 1) / k) > (long long)BS_GROUP_ROWS * nseg * 9 / 10) k++;
    gps[b] = k;
  }
  std::vector<Part> parts((size_t)nstrip * nseg);
  parallel_for(nstrip, [&](long long b0, long long b1) {
    std::vector<int> uc, up;             // a unit's columns, descending; its entries
    for (long long b = b0; b < b1; b++) {
      const int a = I.bstart[b], e = I.bstart[b + 1];
      // units of the strip (runs of one node's rows in one segment, at most 3)
      std::vector<int> ustart, uof(e - a);
      for (int i = a; i < e; i++) {
        const bool same = i > a && group && (*group)[i] == (*group)[i - 1] &&
                          segof(i) == segof(i - 1) && i - ustart.back() < 3;
        if (!same) ustart.push_back(i);
        uof[i - a] = (int)ustart.size() - 1;
      }
      auto inblock = [&](int i, int c) { return c >= a && c < e && segof(c) == segof(i); };
      // rows [u0, u1) with one set of columns (the rows of a node): row u0 stands for them
      auto one_set = [&](int u0, int u1) {
        for (int i = u0 + 1; i < u1; i++)
          if (rp[i + 1] - rp[i] != rp[u0 + 1] - rp[u0] ||
              !std::equal(scol.begin() + rp[u0], scol.begin() + rp[u0 + 1], scol.begin() + rp[i]))
            return false;
        return true;
      };
      // columns of rows [u0, u1) outside them, in the block, on one side
      auto unit_cols = [&](int u0, int u1, bool lower, bool one) {
        uc.clear();
        for (int i = u0; i < (one ? u0 + 1 : u1); i++) {
          const int* b = scol.data() + rp[i];
          const int* e = scol.data() + rp[i + 1];
          if (lower) e = std::lower_bound(b, e, u0); else b = std::lower_bound(b, e, u1);
          for (const int* c = e; c-- > b;)
            if (inblock(i, *c)) uc.push_back(*c);
        }
        if (!one) {
          std::sort(uc.begin(), uc.end(), std::greater<int>());
          uc.erase(std::unique(uc.begin(), uc.end()), uc.end());
        }
        return (int)uc.size();
      };
      // a unit of more columns than BS_MAXW becomes single-row units (a row has at most 127)
      {
        std::vector<int> us2;
        bool split = false;
        for (size_t U = 0; U < ustart.size(); U++) {
          const int u0 = ustart[U], u1 = U + 1 < ustart.size() ? ustart[U + 1] : e;
          if (one_set(u0, u1) || (unit_cols(u0, u1, true, false) <= BS_MAXW &&
                                  unit_cols(u0, u1, false, false) <= BS_MAXW)) {
            us2.push_back(u0);
          } else {
            split = true;
            for (int i = u0; i < u1; i++) us2.push_back(i);
          }
        }
        if (split) {
          ustart.swap(us2);
          for (size_t U = 0; U < ustart.size(); U++) {
            const int u1 = U + 1 < ustart.size() ? ustart[U + 1] : e;
            for (int i = ustart[U]; i < u1; i++) uof[i - a] = (int)U;
          }
        }
      }
      const int nu = (int)ustart.size();
      ustart.push_back(e);
      // unit levels and slots (log2), lower and upper
      std::vector<int> ulev[2] = { std::vector<int>(nu, 0), std::vector<int>(nu, 0) };
      std::vector<unsigned char> ulg[2] = { std::vector<unsigned char>(nu, 0),
                                            std::vector<unsigned char>(nu, 0) };
      std::vector<unsigned char> uone(nu);
      for (int U = 0; U < nu; U++) uone[U] = one_set(ustart[U], ustart[U + 1]);
      for (int t = 0; t < 2; t++)
        for (int k = 0; k < nu; k++) {
          const int U = t == 0 ? k : nu - 1 - k;
          const int w = unit_cols(ustart[U], ustart[U + 1], t == 0, uone[U]);
          for (int c : uc) ulev[t][U] = std::max(ulev[t][U], ulev[t][uof[c - a]] + 1);
          while ((16 << ulg[t][U]) < w) ulg[t][U]++;
        }
      // units of every group of segments
      const int ng = gps[b];
      std::vector<std::vector<int>> grpu(ng);
      std::vector<int> segrows(nseg, 0);
      for (int U = 0; U < nu; U++) {
        const int g = segof(ustart[U]);
        grpu[(long long)g * ng / nseg].push_back(U);
        segrows[g] += ustart[U + 1] - ustart[U];
      }
      const bool wide_block = *std::max_element(segrows.begin(), segrows.end()) > BS_ROWS;
      for (int g = 0; g < ng; g++) {
        Part& P = parts[(size_t)b * nseg + g];
        std::vector<int>& us = grpu[g];
        if (us.empty()) continue;
        int m = 0;
        for (int U : us) m += ustart[U + 1] - ustart[U];
        if (wide_block || m > BS_GROUP_ROWS) { P.fits = false; continue; }
        // by level, then falling slot count, then unit index; local positions follow the
        // lower order
        std::vector<int> ord[2] = { us, us };
        for (int t = 0; t < 2; t++)
          std::stable_sort(ord[t].begin(), ord[t].end(), [&](int x, int y) {
            return ulev[t][x] != ulev[t][y] ? ulev[t][x] < ulev[t][y] : ulg[t][x] > ulg[t][y];
          });
        std::vector<int> upos(nu, -1), uidx(nu, -1);
        for (int k = 0; k < (int)ord[0].size(); k++) {
          const int U = ord[0][k];
          upos[U] = (int)P.rows.size();
          uidx[U] = k;
          for (int i = ustart[U]; i < ustart[U + 1]; i++) P.rows.push_back(i);
        }
        auto pos = [&](int c) { return upos[uof[c - a]] + (c - ustart[uof[c - a]]); };
        for (int t = 0; t < 2; t++) {
          const bool lower = t == 0;
          std::vector<uint2>& desc = P.desc[t];
          std::vector<unsigned short>& col = P.col[t];
          std::vector<int>& src = P.src[t];
          col.assign(4, 0);                    // the zero groups
          src.assign(12, -1);
          desc.assign(1, uint2{ 0u, 0u });     // the empty slot
          int cur = -1, nrow = 0, npair = 0, nslot = 0;
          P.usrc[t].assign(8 * ord[t].size(), -1);
          if (!lower) P.dsrc.assign(4 * ord[t].size(), -1);
          for (int U : ord[t]) {
            const int r0 = ustart[U], nr = ustart[U + 1] - r0;
            const int ns = 1 << ulg[t][U];
            P.lgmax[t] = std::max(P.lgmax[t], (int)ulg[t][U]);
            const int w = unit_cols(r0, r0 + nr, lower, uone[U]);
            // CSR positions of the unit's entries, row by row in the order of uc; a row's
            // entries in pairs, at least one
            up.assign((size_t)nr * w, -1);
            int pairs = 0;
            for (int j = 0; j < nr; j++) {
              const int* b = scol.data() + rp[r0 + j];
              const int* c = scol.data() + rp[r0 + j + 1];
              int k = 0;
              for (int x = 0; x < w; x++) {            // both descending
                while (c > b && c[-1] > uc[x]) c--;
                if (c > b && c[-1] == uc[x]) {
                  up[(size_t)j * w + x] = rp[r0 + j] + (int)spos[c - 1 - scol.data()];
                  k++;
                }
              }
              pairs += std::max(1, (k + 1) / 2);
            }
            if (ulev[t][U] != cur || nslot + ns > BS_SLOTS || nrow + nr > cap_rows ||
                npair + pairs > cap_pairs) {
              P.tab[t].push_back((unsigned)desc.size());
              P.npass[t]++;
              cur = ulev[t][U]; nrow = 0; npair = 0; nslot = 0;
            }
            const int ngroups = (w + 3) / 4;
            const size_t cg0 = col.size() / 4, vg0 = src.size() / 4;
            for (int k = 0; k < 4 * ngroups; k++)  // padding: the zero slot, value zero
              col.push_back((unsigned short)(k < w ? 8 * (pos(uc[k]) + 1) : 0));
            for (int gq = 0; gq < ngroups; gq++)
              for (int j = 0; j < nr; j++)
                for (int k = 4 * gq; k < 4 * gq + 4; k++) src.push_back(k < w ? up[(size_t)j * w + k] : -1);
            if (col.size() / 4 > BS_CM || src.size() / 4 > BS_VM) P.fits = false;
            for (int j = 0; j < ns; j++) {
              // a slot without columns takes the zero groups
              const int ng = std::max(0, std::min(4, ngroups - 4 * j));
              const size_t v0 = ng > 0 ? vg0 + (size_t)4 * j * nr : 0, c0 = ng > 0 ? cg0 + 4 * j : 0;
              desc.push_back(uint2{ (unsigned)(v0 & BS_VM) | (unsigned)upos[U] << 18 |
                                        (unsigned)std::max(0, ng - 1) << 30,
                                    (unsigned)(c0 & BS_CM) | (unsigned)uidx[U] << 16 |
                                        (unsigned)nr << 28 | (unsigned)ulg[t][U] << 30 });
            }
            // row q's couplings inside the unit: lower (l_q0, l_q1), upper (u_q1, u_q2)
            int* us = &P.usrc[t][8 * (size_t)uidx[U]];
            for (int j = 0; j < nr; j++)
              for (int k = 0; k < 2; k++) {
                const int o = lower ? k : k + 1;
                if (o < nr && (lower ? o < j : o > j)) us[2 * j + k] = find(r0 + j, r0 + o);
              }
            if (!lower)
              for (int j = 0; j < nr; j++) P.dsrc[4 * (size_t)uidx[U] + j] = rp[r0 + j];
            nrow += nr;
            npair += pairs;
            nslot += ns;
          }
          // the end, repeated for the entries read past the last pass
          P.tab[t].resize(P.tab[t].size() + 4 * BS_DEPTH, (unsigned)desc.size());
        }
      }
    }
  });
  long long nb = 0, ncg[2] = {0, 0}, nvg[2] = {0, 0}, npass = 0, nunit = 0, nslots = 0, ntab = 0;
  size_t lds = 0;
  for (const Part& P : parts) {
    if (!P.fits) return;
    if (P.rows.empty()) continue;
    nb++;
    for (int t = 0; t < 2; t++) {
      ncg[t] += P.col[t].size() / 4;
      nvg[t] += P.src[t].size() / 4;
      nslots += P.desc[t].size();
      npass += P.npass[t];
      ntab += P.tab[t].size();
    }
    nunit += P.usrc[0].size() / 8;
    lds = std::max(lds, 8 * (P.rows.size() + 3));
  }
  const long long lim = INT_MAX - BS_PAD;
  if (nb == 0 || std::max({ 4 * ncg[0], 4 * ncg[1], nvg[0], nvg[1], nslots, ntab }) > lim) return;
  std::vector<int4> info(4 * nb);
  std::vector<int> gidx(n);
  std::vector<int> src[2], usrc[2], dsrc((size_t)4 * nunit, -1);
  std::vector<unsigned short> col[2];
  std::vector<uint2> desc(nslots);
  std::vector<unsigned> tab(ntab + 64, 0u);
  for (int t = 0; t < 2; t++) {
    src[t].assign(4 * ((size_t)nvg[t] + BS_PAD), -1);
    col[t].assign(4 * ((size_t)ncg[t] + BS_PAD), 0);
    usrc[t].assign((size_t)8 * nunit, -1);
  }
  long long k = 0, rb = 0, sb = 0, tb = 0, ub = 0, cg[2] = {0, 0}, vg[2] = {0, 0};
  for (const Part& P : parts) {
    if (P.rows.empty()) continue;
    const int m = (int)P.rows.size();
    const int su = (int)(sb + P.desc[0].size());
    info[4 * k] = int4{ (int)rb, m, (int)ub, (int)tb };
    info[4 * k + 1] = int4{ P.npass[0], (int)sb, P.npass[1], su };
    info[4 * k + 2] = int4{ (int)vg[0], (int)cg[0], (int)vg[1], (int)cg[1] };
    info[4 * k + 3] = int4{ P.lgmax[0], P.lgmax[1], 0, 0 };
    std::copy(P.rows.begin(), P.rows.end(), gidx.begin() + rb);
    for (int t = 0; t < 2; t++) {
      std::copy(P.tab[t].begin(), P.tab[t].end(), tab.begin() + tb);
      tb += P.tab[t].size();
      std::copy(P.desc[t].begin(), P.desc[t].end(), desc.begin() + sb);
      sb += P.desc[t].size();
      std::copy(P.col[t].begin(), P.col[t].end(), col[t].begin() + 4 * cg[t]);
      std::copy(P.src[t].begin(), P.src[t].end(), src[t].begin() + 4 * vg[t]);
      std::copy(P.usrc[t].begin(), P.usrc[t].end(), usrc[t].begin() + 8 * ub);
      cg[t] += P.col[t].size() / 4;
      vg[t] += P.src[t].size() / 4;
    }
    std::copy(P.dsrc.begin(), P.dsrc.end(), dsrc.begin() + 4 * ub);
    k++; rb += m; ub += P.usrc[0].size() / 8;
  }
  lds_from_zero(k_block_sweep<float>, k_block_sweep<double>);
  B.nb = (int)nb; B.lds = (lds + 15) & ~(size_t)15;
  B.ne_lo = std::count_if(src[0].begin(), src[0].end(), [](int q) { return q >= 0; });
  B.ne_up = std::count_if(src[1].begin(), src[1].end(), [](int q) { return q >= 0; });
  B.npass = npass; B.nunit = nunit; B.nslot = nslots; B.ncol = 4 * (ncg[0] + ncg[1]);
  B.info.upload(info, s); B.gidx.upload(gidx, s); B.tab.upload(tab, s); B.desc.upload(desc, s);
  B.clo.upload(col[0], s); B.cup.upload(col[1], s);
  B.slo.upload(src[0], s); B.sup.upload(src[1], s);
  B.sulo.upload(usrc[0], s); B.suup.upload(usrc[1], s); B.sdg.upload(dsrc, s);
  HIPCHECK(hipStreamSynchronize(s));
  B.on = true;
  if (getenv("RMX_DEBUG"))
    fprintf(stderr, "[rmx] block sweeps: %lld groups of blocks, %lld nodes, %lld + %lld entries (%lld + "
            "%lld padded), %.1f passes per group, %zu bytes LDS\n", nb, nunit, B.ne_lo, B.ne_up,
            4 * nvg[0], 4 * nvg[1], (double)npass / nb, B.lds);
}

// Node sweep layout (k_node_sweep) of one triangle over all strips.  Units are those of
// build_blocks (runs of rows of one node in one segment, at most 3); a unit's columns lie in
// its rows' strip and segment.  Units are scheduled by levels, as early or as late as their
// dependencies allow, whichever keeps fewer rows alive; a unit's LDS places are free again
// after the last level that reads them.  Off when a strip's live rows do not fit LDS.
static void build_nodes(NodeSweep& S, const Ilu& I, bool lower, const std::vector<int>* group,
                        const std::vector<int>& scol, const std::vector<unsigned char>& spos,
                        hipStream_t s)
{
  S.on = false;
  const int n = I.n, nstrip = I.nblk;
  const std::vector<int>& rp = I.h_rp;
  if (I.nnz >= (1LL << 29) || n >= (1 << 30) - 64) return;
  const bool sg = !I.seg.empty();
  auto segof = [&](int i) { return sg ? I.seg[i] : 0; };
  // units, ascending rows; the strip of every unit
  std::vector<int> ustart, uof(n), ustrip, ub(nstrip + 1, 0);
  auto one_set = [&](int u0, int u1) {          // one set of columns: row u0 stands for all
    for (int i = u0 + 1; i < u1; i++)
      if (rp[i + 1] - rp[i] != rp[u0 + 1] - rp[u0] ||
          !std::equal(scol.begin() + rp[u0], scol.begin() + rp[u0 + 1], scol.begin() + rp[i]))
        return false;
    return true;
  };
  for (int b = 0; b < nstrip; b++) {
    ub[b] = (int)ustart.size();
    for (int i = I.bstart[b]; i < I.bstart[b + 1];) {
      int j = i + 1;
      while (j < I.bstart[b + 1] && group && (*group)[j] == (*group)[i] && segof(j) == segof(i) &&
             j < i + 3) j++;
      // rows of different columns, which could be more than a unit takes: single rows
      if (j > i + 1 && !one_set(i, j)) {
        int w = 0;
        for (int k = i; k < j; k++) w += rp[k + 1] - rp[k];
        if (w > BS_MAXW) j = i + 1;
      }
      for (int k = i; k < j; k++) uof[k] = (int)ustart.size();
      ustart.push_back(i);
      ustrip.push_back(b);
      i = j;
    }
  }
  const int nu = (int)ustart.size();
  ub[nstrip] = nu;
  ustart.push_back(n);
  std::vector<unsigned char> uone(nu), ulg(nu, 0);
  std::vector<int> uw(nu, 0);
  // columns of a unit, descending (uc), and the units they belong to
  auto cols_of = [&](int U, std::vector<int>& uc) {
    const int u0 = ustart[U], u1 = ustart[U + 1], a = I.bstart[ustrip[U]], e = I.bstart[ustrip[U] + 1];
    uc.clear();
    for (int i = u0; i < (uone[U] ? u0 + 1 : u1); i++) {
      const int* b = scol.data() + rp[i];
      const int* z = scol.data() + rp[i + 1];
      if (lower) { z = std::lower_bound(b, z, u0); b = std::lower_bound(b, z, a); }
      else { b = std::lower_bound(b, z, u1); z = std::lower_bound(b, z, e); }
      for (const int* c = z; c-- > b;)
        if (!sg || segof(*c) == segof(i)) uc.push_back(*c);
    }
    if (!uone[U]) {
      std::sort(uc.begin(), uc.end(), std::greater<int>());
      uc.erase(std::unique(uc.begin(), uc.end()), uc.end());
    }
  };
  // the units that a unit reads, their number if `out` is null
  auto units = [&](const std::vector<int>& uc, int* out) {
    int last = -1, k = 0;
    for (int c : uc)
      if (uof[c] != last) { last = uof[c]; if (out) out[k] = last; k++; }
    return k;
  };
  std::vector<long long> dp(nu + 1, 0);
  parallel_for(nu, [&](long long u0, long long u1) {
    std::vector<int> uc;
    for (long long U = u0; U < u1; U++) {
      uone[U] = one_set(ustart[U], ustart[U + 1]);
      cols_of((int)U, uc);
      uw[U] = (int)uc.size();
      while ((16 << ulg[U]) < uw[U]) ulg[U]++;
      dp[U + 1] = units(uc, nullptr);
    }
  });
  for (int U = 0; U < nu; U++) dp[U + 1] += dp[U];
  std::vector<int> dep(dp[nu]);
  if (dp[nu] > 0) parallel_for(nu, [&](long long u0, long long u1) {
    std::vector<int> uc;
    for (long long U = u0; U < u1; U++) { cols_of((int)U, uc); units(uc, dep.data() + dp[U]); }
  });
  std::vector<int> place(nu, 0), order(nu), nlev(nstrip, 0), live(nstrip, 1), lbeg;
  std::vector<std::vector<int>> lptr(nstrip);    // level offsets of a strip into its order
  parallel_for(nstrip, [&](long long b0, long long b1) {
    for (long long b = b0; b < b1; b++) {
      const int a = ub[b], e = ub[b + 1], m = e - a;
      if (m == 0) { lptr[b].assign(1, 0); continue; }
      std::vector<int> lev[2] = { std::vector<int>(m, 0), std::vector<int>(m, INT_MAX) };
      int L = 0;
      for (int k = 0; k < m; k++) {
        const int U = lower ? a + k : e - 1 - k;
        int l = 0;
        for (long long q = dp[U]; q < dp[U + 1]; q++) l = std::max(l, lev[0][dep[q] - a] + 1);
        lev[0][U - a] = l;
        L = std::max(L, l + 1);
      }
      for (int k = m - 1; k >= 0; k--) {
        const int U = lower ? a + k : e - 1 - k;
        int& l = lev[1][U - a];
        if (l == INT_MAX) l = lev[0][U - a];     // nothing reads it
        for (long long q = dp[U]; q < dp[U + 1]; q++)
          lev[1][dep[q] - a] = std::min(lev[1][dep[q] - a], l - 1);
      }
      // order by level, a level's units by falling slot count (aligned to their number); LDS
      // places as a linear scan gives them
      std::vector<int> best, bplace, bptr;
      for (int t = 0; t < 2; t++) {
        const std::vector<int>& lv = lev[t];
        std::vector<int> last(lv), ptr(4 * (size_t)L + 1, 0), ord(m), dptr(L + 1, 0), dl(m), pl(m);
        for (int U = a; U < e; U++)
          for (long long q = dp[U]; q < dp[U + 1]; q++)
            last[dep[q] - a] = std::max(last[dep[q] - a], lv[U - a]);
        for (int k = 0; k < m; k++) { ptr[4 * lv[k] + 3 - ulg[a + k] + 1]++; dptr[last[k] + 1]++; }
        for (int l = 0; l < 4 * L; l++) ptr[l + 1] += ptr[l];
        for (int l = 0; l < L; l++) dptr[l + 1] += dptr[l];
        std::vector<int> lp(L + 1);
        for (int l = 0; l <= L; l++) lp[l] = ptr[4 * l];
        {
          std::vector<int> f(ptr), g(dptr);
          for (int k = 0; k < m; k++) { ord[f[4 * lv[k] + 3 - ulg[a + k]]++] = k; dl[g[last[k]]++] = k; }
        }
        std::vector<int> freed[4];
        int top = 1;
        for (int l = 0; l < L; l++) {
          for (int q = lp[l]; q < lp[l + 1]; q++) {
            const int k = ord[q], w = ustart[a + k + 1] - ustart[a + k];
            if (!freed[w].empty()) { pl[k] = freed[w].back(); freed[w].pop_back(); }
            else { pl[k] = top; top += w; }
          }
          for (int q = dptr[l]; q < dptr[l + 1]; q++)
            freed[ustart[a + dl[q] + 1] - ustart[a + dl[q]]].push_back(pl[dl[q]]);
        }
        if (t == 0 || top < live[b]) { live[b] = top; best.swap(ord); bplace.swap(pl); bptr.swap(lp); }
      }
      for (int k = 0; k < m; k++) { order[a + k] = a + best[k]; place[a + k] = bplace[k]; }
      lptr[b].swap(bptr);
      nlev[b] = L;
    }
  });
  // waves: the fewest that hold an average level in one pass (lower + upper sweep, FP64, 1 / 2 /
  // 4 / 8 waves: 30 slots a level 842 / 554 / 517 / 816 us, 11 slots 627 / 399 / 575 / 935, 59 and
  // 54 slots 5.3 / 3.5 / 3.2 / 3.7 ms, 104 slots 21 / 14.3 / 14.6 / 15.3 ms): at most four, past
  // which a pass takes longer by what it saves in passes
  long long slots = 0, levels = 0;
  int lgmax = 0, maxlive = 1;
  for (int U = 0; U < nu; U++) { slots += 1 << ulg[U]; lgmax = std::max(lgmax, (int)ulg[U]); }
  for (int b = 0; b < nstrip; b++) { levels += nlev[b]; maxlive = std::max(maxlive, live[b]); }
  S.lds = 8 * ((size_t)maxlive + 2);
  if (maxlive > 65533 || S.lds > (size_t)NS_LDS) return;
  S.waves = 1;
  while (S.waves < NS_WAVES && 16LL * S.waves * levels < slots) S.waves *= 2;
  if (const char* e = getenv("RMX_NODE_WAVES")) S.waves = std::max(1, std::min(NS_WAVES, atoi(e)));
  const int cap = 16 * S.waves;
  // passes, and where every unit's slots, column groups and row groups start (descriptor 0 of
  // a strip is empty; column group 0 and row groups 0 to 2 are zero)
  std::vector<int4> info(nstrip);
  std::vector<unsigned> tab;
  std::vector<unsigned> us0(nu), uc0(nu), uv0(nu);
  long long nd = 0, nc = 1, nv = 3;
  for (int b = 0; b < nstrip; b++) {
    const long long d0 = nd++;
    const size_t t0 = tab.size();
    for (int l = 0; l < nlev[b]; l++) {
      int ns = cap;
      for (int q = lptr[b][l]; q < lptr[b][l + 1]; q++) {
        const int U = order[ub[b] + q], ng = (uw[U] + 3) / 4;
        if (ns + (1 << ulg[U]) > cap) { tab.push_back((unsigned)(nd - d0)); ns = 0; }
        ns += 1 << ulg[U];
        us0[U] = (unsigned)nd; uc0[U] = (unsigned)nc; uv0[U] = (unsigned)nv;
        nd += 1 << ulg[U];
        nc += ng;
        nv += (long long)ng * (ustart[U + 1] - ustart[U]);
      }
    }
    info[b] = int4{ (int)(tab.size() - t0), (int)t0, (int)d0, 0 };
    tab.resize(tab.size() + 4 * NS_DEPTH, (unsigned)(nd - d0));   // repeated past the last pass
  }
  if (nd >= INT_MAX || nv >= (1 << 30) - BS_PAD) return;
  const size_t npass = tab.size() - (size_t)nstrip * 4 * NS_DEPTH;
  tab.resize(tab.size() + 64, 0u);
  std::vector<uint4> desc(nd, uint4{ 0u, 0u, 0u, 0u });
  std::vector<unsigned short> col(4 * (size_t)(nc + BS_PAD), 0);
  std::vector<int> src(4 * (size_t)(nv + BS_PAD), -1), wsrc(2 * (size_t)n, -1);
  parallel_for(nu, [&](long long a, long long z) {
    std::vector<int> uc;
    auto find = [&](int r, int c) {
      const auto b = scol.begin() + rp[r], e = scol.begin() + rp[r + 1];
      const auto it = std::lower_bound(b, e, c);
      return it != e && *it == c ? rp[r] + (int)spos[it - scol.begin()] : -1;
    };
    for (long long U = a; U < z; U++) {
      const int r0 = ustart[U], nr = ustart[U + 1] - r0;
      cols_of((int)U, uc);
      const int w = (int)uc.size(), ng = (w + 3) / 4;
      for (int k = 0; k < w; k++)
        col[4 * (size_t)uc0[U] + k] = (unsigned short)(place[uof[uc[k]]] + (uc[k] - ustart[uof[uc[k]]]));
      for (int j = 0; j < nr; j++) {
        const int* b = scol.data() + rp[r0 + j];
        const int* c = scol.data() + rp[r0 + j + 1];
        for (int k = 0; k < w; k++) {              // both descending
          while (c > b && c[-1] > uc[k]) c--;
          if (c > b && c[-1] == uc[k])
            src[4 * (size_t)uv0[U] + ((size_t)(k / 4) * nr + j) * 4 + k % 4] =
                rp[r0 + j] + (int)spos[c - 1 - scol.data()];
        }
      }
      for (int j = 0; j < (1 << ulg[U]); j++) {
        const int g = std::max(0, std::min(4, ng - 4 * j));
        desc[us0[U] + j] = uint4{ (g ? uv0[U] + (unsigned)(4 * j * nr) : 0u) | (unsigned)nr << 30,
                                  (g ? uc0[U] + (unsigned)(4 * j) : 0u) | (unsigned)std::max(0, g - 1) << 30,
                                  (unsigned)r0 | (unsigned)ulg[U] << 30, (unsigned)place[U] };
      }
      for (int j = 0; j < nr; j++)                 // as in build_blocks
        for (int k = 0; k < 2; k++) {
          const int o = lower ? k : k + 1;
          if (o < nr && (lower ? o < j : o > j)) wsrc[2 * (size_t)(r0 + j) + k] = find(r0 + j, r0 + o);
        }
    }
  });
  lds_from_zero(k_node_sweep<float, true, 0>, k_node_sweep<float, true, 1>, k_node_sweep<float, true, 2>,
                k_node_sweep<float, false, 0>, k_node_sweep<float, false, 1>, k_node_sweep<float, false, 2>,
                k_node_sweep<double, true, 0>, k_node_sweep<double, true, 1>, k_node_sweep<double, true, 2>,
                k_node_sweep<double, false, 0>, k_node_sweep<double, false, 1>,
                k_node_sweep<double, false, 2>);
  S.lgmax = std::min(2, lgmax);
  S.info.upload(info, s); S.tab.upload(tab, s); S.desc.upload(desc, s);
  S.cols.upload(col, s); S.src.upload(src, s); S.wsrc.upload(wsrc, s);
  HIPCHECK(hipStreamSynchronize(s));
  S.on = true;
  if (getenv("RMX_DEBUG"))
    fprintf(stderr, "[rmx] %s node sweep: %d strip(s), %d nodes, %lld slots, %lld levels, %zu "
            "passes, %d waves, %d LDS places\n", lower ? "lower" : "upper", nstrip, nu, slots,
            levels, npass, S.waves, maxlive);
}

// Segment of every row: each strip [bstart[b], bstart[b+1]) is cut into nseg parts of
// about equal row count along the principal axis of its nodes' coordinates (across the
// channel for a strip of cross-sections); a node's rows share a segment.
std::vector<int> cut_segments(const std::vector<int>& bstart, const std::vector<int>& group,
                              const HostModel& hm, int nseg)
{
  const int nblk = (int)bstart.size() - 1;
  std::vector<int> seg(bstart[nblk], 0);
  parallel_for(nblk, [&](long long b0, long long b1) {
    std::vector<std::pair<double, int>> proj;
    for (long long b = b0; b < b1; b++) {
      const int a = bstart[b], e = bstart[b + 1];
      if (e <= a) continue;
      double mx = 0, my = 0;
      for (int i = a; i < e; i++) { mx += hm.x[group[i]]; my += hm.y[group[i]]; }
      mx /= (e - a); my /= (e - a);
      double sxx = 0, sxy = 0, syy = 0;
      for (int i = a; i < e; i++) {
        const double dx = hm.x[group[i]] - mx, dy = hm.y[group[i]] - my;
        sxx += dx * dx; sxy += dx * dy; syy += dy * dy;
      }
      // eigenvector of the larger eigenvalue of [[sxx, sxy], [sxy, syy]]
      const double th = 0.5 * std::atan2(2.0 * sxy, sxx - syy);
      const double ex = std::cos(th), ey = std::sin(th);
      proj.clear();
      for (int i = a; i < e; i++)
        proj.emplace_back((hm.x[group[i]] - mx) * ex + (hm.y[group[i]] - my) * ey, i);
      std::sort(proj.begin(), proj.end());
      // equal row counts, cuts moved to the next node so a node's rows share a segment
      const int m = e - a;
      int k = 0;
      for (int t = 0; t < m; t++) {
        if (k + 1 < nseg && t >= (long long)m * (k + 1) / nseg && t > 0 &&
            group[proj[t].second] != group[proj[t - 1].second] && proj[t].first != proj[t - 1].first)
          k++;
        seg[proj[t].second] = k;
      }
    }
  });
  return seg;
}

// Chunk layout of every block (host); false where a block has more than BS_ROWS rows, or there
// are more than CH_BLOCKS blocks.
bool chunk_layout(const Ilu& I, ChunkLayout& L)
{
  const int n = I.n, nseg = std::max(1, I.nseg), nb = I.nblk * nseg;
  const std::vector<int>& rp = I.h_rp;
  auto segof = [&](int i) { return I.seg.empty() ? 0 : I.seg[i]; };
  // rows of every block, ascending
  std::vector<int> blk(n), start(nb + 1, 0), rows(n), at(n);
  for (int b = 0; b < I.nblk; b++)
    for (int i = I.bstart[b]; i < I.bstart[b + 1]; i++) start[(blk[i] = b * nseg + segof(i)) + 1]++;
  int most = 0;
  for (int b = 0; b < nb; b++) most = std::max(most, start[b + 1]);
  if (most > BS_ROWS || nb > CH_BLOCKS) return false;
  for (int b = 0; b < nb; b++) start[b + 1] += start[b];
  {
    std::vector<int> next(start.begin(), start.end() - 1);
    for (int i = 0; i < n; i++) { at[i] = next[blk[i]] - start[blk[i]]; rows[next[blk[i]]++] = i; }
  }
  std::vector<int> cbase(nb + 1, 0);
  for (int b = 0; b < nb; b++) cbase[b + 1] = cbase[b] + (start[b + 1] - start[b] + CH_ROWS - 1) / CH_ROWS;
  const int nch = cbase[nb];
  std::vector<int> slot(n);
  std::vector<int4> chunks(nch);
  std::vector<unsigned char> cdesc[2] = { std::vector<unsigned char>(nch), std::vector<unsigned char>(nch) };
  std::vector<unsigned> idx[2];
  std::vector<int> src[2], pbase[2] = { std::vector<int>(nb + 1, 0), std::vector<int>(nb + 1, 0) };
  std::vector<long long> ne(nb, 0);
  for (int pass = 0; pass < 2; pass++) {            // count packets, then fill
    parallel_for(nb, [&](long long b0, long long b1) {
      std::vector<std::pair<int, int>> e[CH_ROWS];  // column's place, CSR position
      for (int b = (int)b0; b < (int)b1; b++) {
        const int m = start[b + 1] - start[b], k1 = cbase[b + 1] - cbase[b];
        for (int dir = 0; dir < 2; dir++) {
          int pk = 0;
          for (int t = 0; t < k1; t++) {
            const int k = dir ? k1 - 1 - t : t;
            size_t w = 0;
            for (int c = 0; c < CH_ROWS; c++) {
              const int pos = CH_ROWS * k + (dir ? CH_ROWS - 1 - c : c);
              e[c].clear();
              if (pos >= m) continue;
              const int i = rows[start[b] + pos];
              if (pass == 0 && dir == 0) slot[i] = (cbase[b] + k) * CH_ROWS + c;
              for (int p = rp[i] + 1; p < rp[i + 1]; p++) {
                const int j = I.h_cols[p];
                if (blk[j] != b || (dir ? j < i : j > i) || at[j] / CH_ROWS == k) continue;
                e[c].emplace_back(at[j], p);
              }
              w = std::max(w, (e[c].size() + 3) / 4);
            }
            const int np = std::max(1, (int)(w + 1) / 2);
            if (pass == 1) {
              const size_t p0 = (size_t)pbase[dir][b] + pk;
              cdesc[dir][cbase[b] + t] = (unsigned char)np;
              for (int c = 0; c < CH_ROWS; c++) {
                std::sort(e[c].begin(), e[c].end());
                ne[b] += (long long)e[c].size();
                const unsigned own = 8u * (CH_ROWS * k + (dir ? CH_ROWS - 1 - c : c));
                for (int p = 0; p < np; p++)
                  for (int q = 0; q < 4; q++) {
                    unsigned o[2] = { own, own };
                    int from[2] = { -1, -1 };
                    for (int h = 0; h < 2; h++) {
                      const size_t l = 4 * (2 * p + h) + q;
                      if (l < e[c].size()) { o[h] = 8u * e[c][l].first; from[h] = e[c][l].second; }
                    }
                    const size_t lane = (p0 + p) * 64 + 4 * c + q;
                    idx[dir][lane] = o[0] | o[1] << 16;
                    src[dir][2 * lane] = from[0];
                    src[dir][2 * lane + 1] = from[1];
                  }
              }
              if (dir == 0)
                chunks[cbase[b] + k] = int4{ start[b] + CH_ROWS * k, std::min(CH_ROWS, m - CH_ROWS * k),
                                             cbase[b] + k, cbase[b] + k1 - 1 - k };
            }
            pk += np;
          }
          // the loads ahead of the last chunks end in packets of zeros times the block's first row,
          // not in the next block's, whose columns may lie past this block's rows
          if (pass == 0) pbase[dir][b + 1] = pk + CH_PK;
        }
      }
    });
    if (pass == 0)
      for (int dir = 0; dir < 2; dir++) {
        for (int b = 0; b < nb; b++) pbase[dir][b + 1] += pbase[dir][b];
        idx[dir].assign((size_t)pbase[dir][nb] * 64, 0);
        src[dir].assign((size_t)pbase[dir][nb] * 128, -1);
      }
  }
  for (int b = 0; b < nb; b++)
    if (start[b + 1] > start[b]) {
      L.info.push_back(int4{ start[b], start[b + 1] - start[b], cbase[b], 0 });
      L.info.push_back(int4{ pbase[0][b], pbase[1][b], 0, 0 });
    }
  // loaded ahead: two packets where at most a tenth of the chunks has more (their others are then
  // loaded when they are due), else four.  FP32, us with two and with four: rows of up to 16 entries
  // a side, 2,047 of them, 68 and 80, 700 of them 26 and 30; meanders of 231,000 and 923,000 rows
  // (below the tenth) 39 and 39, 70 and 70; channels of 36,000 and 145,000 rows (above it) 36 and 34,
  // 46 and 39, quadrilaterals of 5,600 rows 39 and 35, 1.8 million rows 143 and 140.
  long long over = 0;
  for (int dir = 0; dir < 2; dir++)
    for (unsigned char np : cdesc[dir]) over += np > 2;
  L.ahead = over * 20 > 2LL * nch ? CH_PK : 2;
  L.nch = nch;
  L.most = most;
  for (long long v : ne) L.ne += v;
  L.rows.swap(rows);
  L.slot.swap(slot);
  L.chunks.swap(chunks);
  for (int dir = 0; dir < 2; dir++) {
    L.cnt[dir].swap(cdesc[dir]);
    L.idx[dir].swap(idx[dir]);
    L.src[dir].swap(src[dir]);
  }
  return true;
}

// Rows of every block of a layout, and of the places that its sweeps read in LDS, the packets
// loaded past a chunk's own included (as chunk_sweep takes them), one more than the highest.
void chunk_reach(const ChunkLayout& L, std::vector<int>& rows, std::vector<int>& reach)
{
  rows.clear(); reach.clear();
  for (size_t b = 0; 2 * b < L.info.size(); b++) {
    const int m = L.info[2 * b].y, cb = L.info[2 * b].z, nch = (m + CH_ROWS - 1) / CH_ROWS;
    unsigned top = 0;
    for (int dir = 0; dir < 2; dir++) {
      size_t p = dir ? L.info[2 * b + 1].y : L.info[2 * b + 1].x;
      for (int t = 0; t < nch; t++) {
        const int np = L.cnt[dir][cb + t], read = np <= 2 ? 2 : std::max(np, L.ahead);
        for (size_t k = p * 64; k < (p + read) * 64; k++)
          top = std::max({ top, L.idx[dir][k] & 0xFFFFu, L.idx[dir][k] >> 16 });
        p += np;
      }
    }
    rows.push_back(m);
    reach.push_back((int)(top / 8) + 1);
  }
}

static void build_chunks(Ilu& I, hipStream_t s)
{
  ChunkSweep& S = I.cs;
  ChunkLayout L;
  S.on = false;
  if (!chunk_layout(I, L)) return;
  lds_from_zero(k_chunk_sweep<float, 2>, k_chunk_sweep<float, CH_PK>, k_chunk_sweep<double, 2>,
                k_chunk_sweep<double, CH_PK>);
  S.nb = (int)L.info.size() / 2;
  S.ahead = L.ahead;
  S.nch = L.nch;
  S.ne = L.ne;
  S.lds = 8 * (size_t)(((L.most + CH_ROWS - 1) / CH_ROWS) * CH_ROWS + 64);
  S.info.upload(L.info, s);
  S.rows.upload(L.rows, s);
  S.slot.upload(L.slot, s);
  S.chunks.upload(L.chunks, s);
  S.dlo.upload(L.cnt[0], s); S.dup.upload(L.cnt[1], s);
  S.ilo.upload(L.idx[0], s); S.iup.upload(L.idx[1], s);
  S.slo.upload(L.src[0], s); S.sup.upload(L.src[1], s);
  HIPCHECK(hipStreamSynchronize(s));
  S.on = true;
}

// Schedule of the row-by-row factorisation: rows by lower level of the whole pattern, per
// level position {row, start, width, lower entries}, per sorted lower entry the start and
// length (after the diagonal) of its pivot row, and the plan.
static void build_rows(Ilu& I, const std::vector<int>& scol, hipStream_t s)
{
  const int n = I.n;
  std::vector<int> lev(n, 0), fptr, frows;
  levels(0, n, I.h_rp, I.h_cols, true, std::vector<int>(), lev, fptr, frows);
  I.flev = fptr;
  std::vector<int4> desc(n);
  std::vector<int2> piv(I.nnz, int2{0, 0});
  parallel_for(n, [&](long long a, long long e) {
    for (long long w = a; w < e; w++) {
      const int i = frows[w];
      const int p0 = I.h_rp[i], wi = I.h_rp[i + 1] - p0;
      int nk = 0;
      while (nk < wi && scol[p0 + nk] < i) {
        const int k = scol[p0 + nk];
        piv[p0 + nk] = int2{ I.h_rp[k], I.h_rp[k + 1] - I.h_rp[k] - 1 };
        nk++;
      }
      desc[w] = int4{ i, p0, wi, nk };
    }
  });
  // plan offsets: every row's concatenated pivot-row entries
  std::vector<long long> pbase(n + 1, 0);
  for (int w = 0; w < n; w++) {
    long long tot = 0;
    for (int t = 0; t < desc[w].w; t++) tot += piv[desc[w].y + t].y;
    pbase[w + 1] = pbase[w] + tot;
  }
  I.fdesc.upload(desc, s);
  I.fpiv.upload(piv, s);
  I.fpbase.upload(pbase, s);
  I.plan.alloc(std::max<long long>(pbase[n], 1));
  k_ilu_plan<<<n, 64, 0, s>>>(I.fdesc.p, n, I.cols.p, I.srt_cols.p, I.srt_pos.p, I.fpiv.p,
                              I.fpbase.p, I.plan.p);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipStreamSynchronize(s));
}

// Schedule of the factorisation by units of up to `rows_max` rows.  None: a unit of more than
// FP pivot units, or a pattern that couples a unit to some rows of another.
static std::shared_ptr<FlowSchedule> build_units(const Ilu& I, const std::vector<int>& unit,
                                                 int rows_max, const std::vector<int>& scol,
                                                 hipStream_t s)
{
  const int n = I.n;
  const std::vector<int>& rp = I.h_rp;
  std::vector<int> start, of(n);
  for (int i = 0; i < n; i++) {
    const int w = rp[i + 1] - rp[i];
    const bool same = i > 0 && unit[i] == unit[i - 1] && i - start.back() < rows_max &&
                      w == rp[i] - rp[i - 1] &&
                      std::equal(&scol[rp[i]], &scol[rp[i]] + w, &scol[rp[i - 1]]);
    if (!same) start.push_back(i);
    of[i] = (int)start.size() - 1;
  }
  const int nu = (int)start.size();
  start.push_back(n);
  // pivot units, places, levels
  std::vector<int> lst(nu + 1, 0), sd(nu), lev(nu, 0);
  std::vector<int4> piv;
  piv.reserve(rp[n] / 4);
  std::vector<long long> ub(nu + 1, 0);
  int top = 0;
  for (int g = 0; g < nu; g++) {
    const int r0 = start[g], rows = start[g + 1] - r0, p0 = rp[r0], w = rp[r0 + 1] - p0;
    int t = 0;
    while (t < w && scol[p0 + t] < r0) {
      const int K = of[scol[p0 + t]], R = start[K + 1] - start[K];
      for (int q = 0; q < R; q++)
        if (t + q >= w || scol[p0 + t + q] != start[K] + q) return nullptr;
      piv.push_back(int4{ (int)ub[K], t | R << 8, start[K + 1] - 1, K });
      lev[g] = std::max(lev[g], lev[K] + 1);
      t += R;
    }
    for (int q = 0; q < rows; q++)
      if (t + q >= w || scol[p0 + t + q] != r0 + q) return nullptr;
    sd[g] = t;
    top = std::max(top, lev[g]);
    lst[g + 1] = (int)piv.size();
    if (lst[g + 1] - lst[g] > FP) return nullptr;
    ub[g + 1] = ub[g] + (w - t);
  }
  std::vector<int> ptr(top + 2, 0), at(nu);
  for (int g = 0; g < nu; g++) ptr[lev[g] + 1]++;
  for (int l = 0; l <= top; l++) ptr[l + 1] += ptr[l];
  for (int g = 0; g < nu; g++) at[g] = ptr[lev[g]]++;
  std::vector<int4> desc(2 * (size_t)nu);
  long long lines = 0;
  for (int g = 0; g < nu; g++) {
    const int r0 = start[g], p0 = rp[r0], w = rp[r0 + 1] - p0, np = lst[g + 1] - lst[g];
    desc[2 * (size_t)at[g]] = int4{ r0, p0, w | (start[g + 1] - r0) << 8 | np << 16, sd[g] };
    desc[2 * (size_t)at[g] + 1] = int4{ lst[g], (int)lines, (int)ub[g], 0 };
    lines += (long long)np * (w > 64 ? 2 : 1);
  }
  if (lines > INT_MAX || ub[nu] > INT_MAX) return nullptr;
  for (int4& e : piv) e.w = at[e.w];
  if (piv.empty()) piv.push_back(int4{ 0, 0, 0, 0 });
  auto sch = std::make_shared<FlowSchedule>();
  FlowSchedule& F = *sch;
  F.nu = nu;
  F.cols = ub[nu];
  F.desc.upload(desc, s);
  F.list.upload(piv, s);
  F.plan.alloc(64 * (size_t)std::max(lines, 1LL));
  k_unit_plan<<<nu, 64, 0, s>>>(F.desc.p, F.list.p, I.srt_cols.p, F.plan.p);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipStreamSynchronize(s));
  return sch;
}

// Every row's columns ascending, and their places in the row; whether a row has a column twice.
static bool sorted_columns(const std::vector<int>& rp, const std::vector<int>& cl,
                           std::vector<int>& scol, std::vector<unsigned char>& spos)
{
  const int n = (int)rp.size() - 1;
  scol.resize(rp[n]);
  spos.resize(rp[n]);
  for (int i = 0; i < n; i++)
    if (rp[i + 1] - rp[i] > FW) fail(RMX_ERR_RANGE, "ILU(0): row wider than 128 columns");
  std::atomic<bool> twice{false};
  parallel_for(n, [&](long long a, long long b) {
    std::vector<std::pair<int, int>> tmp;
    for (long long i = a; i < b; i++) {
      tmp.clear();
      for (int q = rp[i]; q < rp[i + 1]; q++) tmp.emplace_back(cl[q], q - rp[i]);
      std::sort(tmp.begin(), tmp.end());
      for (size_t t = 0; t < tmp.size(); t++) {
        scol[rp[i] + t] = tmp[t].first;
        spos[rp[i] + t] = (unsigned char)tmp[t].second;
        if (t > 0 && tmp[t].first == tmp[t - 1].first) twice = true;
      }
    }
  });
  return twice;
}

// Strips: contiguous row ranges of about equal size.  With `group` (the node of every
// equation) a cut moves forward to the next row of another node, so the U, V, H equations
// of one node stay in one strip.  level_cap > 0 splits the sweeps' levels into parts of at
// most that many rows.
// `unit`: rows of one unit of the block and node sweeps have one value (the node, or a run of
// rows with one set of columns).  `twin`: an instance of the same pattern and units, whose
// schedule of the factorisation serves this one too.  `twice`: a row has a column more than once,
// whose values add up: only the row-by-row factorisation and the level sweeps take every entry
// of a row by itself.
void ilu_setup(Ilu& I, int n, const std::vector<int>& rp, const std::vector<int>& cl, int nblk,
               const std::vector<int>* group, const std::vector<int>& unit, hipStream_t s,
               const HostModel* hm, int nseg, int level_cap, const std::vector<int>& scol,
               const std::vector<unsigned char>& spos, const Ilu* twin, bool twice)
{
  I.ready = I.fac64 = I.fac32 = false;
  I.n = n;
  I.nblk = std::max(1, std::min(nblk, n));
  I.bstart.assign(I.nblk + 1, 0);
  for (int b = 0; b <= I.nblk; b++) {
    int cut = (int)((long long)n * b / I.nblk);
    if (group && b > 0) {
      cut = std::max(cut, I.bstart[b - 1]);
      while (cut > 0 && cut < n && (*group)[cut] == (*group)[cut - 1]) cut++;
    }
    I.bstart[b] = cut;
  }
  I.bstart[I.nblk] = n;
  // segments: each strip is cut across into nseg parts of equal row count along the
  // principal axis of its nodes' coordinates (across the channel for a strip of
  // cross-sections); entries coupling two segments are left out of the sweeps as well
  I.seg.clear();
  I.nseg = 1;
  if (group && hm && nseg > 1) {
    I.nseg = nseg;
    I.seg = cut_segments(I.bstart, *group, *hm, nseg);
  }
  I.h_rp = rp;
  I.h_cols = cl;
  I.nnz = I.h_rp[n];
  I.rp.upload(I.h_rp, s); I.cols.upload(I.h_cols, s);
  I.srt_cols.upload(scol, s); I.srt_pos.upload(spos, s);
  I.flev.clear();
  I.fdesc.release();
  // units, of single rows where the pattern couples parts of runs, else row by row (single
  // rows, FP64, 36,000 in a band of 8 a side, 4,000 in one of 30: 54 and 6.2 ms, row by row 78
  // and 8.6)
  I.fu.u32.release(); I.fu.u64.release();
  I.fu.sch = twin ? twin->fu.sch : twice ? nullptr : build_units(I, unit, FU, scol, s);
  if (!I.fu.sch && !twin && !twice) I.fu.sch = build_units(I, unit, 1, scol, s);
  if (!I.fu.sch) build_rows(I, scol, s);
  // strip sweeps: a level of more rows than the staged sweep's row groups (512 threads, 4
  // lanes per row) is split, so that no level needs a second round, whose entries would be
  // loaded inside the level instead of one level ahead
  I.level_cap = level_cap;
  if (const char* e = getenv("RMX_LEVEL_CAP")) I.level_cap = std::max(0, atoi(e));
  // strip ILU of few blocks: by chunks; the reference sweeps keep the order of the substitution
  // (and the block sweeps where RMX_SWEEP or their pass caps ask for them)
  I.cs.on = false;
  if (level_cap > 0 && !twice && sweep_variant() != 2 && !getenv("RMX_BLOCK_LEVEL_ROWS") &&
      !getenv("RMX_BLOCK_LEVEL_PAIRS")) build_chunks(I, s);
  I.bs.on = I.nlo.on = I.nup.on = false;
  if (!I.cs.on && !twice) build_blocks(I, &unit, scol, spos, s);
  if (!I.cs.on && !I.bs.on && !twice) {
    // both triangles side by side (their schedules are serial in a strip)
    int dev = 0;
    HIPCHECK(hipGetDevice(&dev));
    auto up = std::async(std::launch::async, [&] {
      HIPCHECK(hipSetDevice(dev));
      build_nodes(I.nup, I, false, &unit, scol, spos, s);
    });
    build_nodes(I.nlo, I, true, &unit, scol, spos, s);
    up.get();
  }
  // the level sweeps where neither runs, or RMX_SWEEP asks for them
  const bool full = !(I.cs.on || I.bs.on || (I.nlo.on && I.nup.on)) || sweep_variant() < 2;
  I.lo.packed = I.up.packed = false;
  I.lo.nlev_max = I.up.nlev_max = -1;
  if (full || I.nlo.on) I.lo.xp.alloc(n);
  if (full) I.up.xp.alloc(n);
  else count_entries(I);
  // forward position (global, concatenated) of the row at each backward position
  if (full) {
    std::vector<int> olo, oup;
    build_sweep(I.lo, I, true, olo, s);
    build_sweep(I.up, I, false, oup, s);
    std::vector<int> fpos(n), f2b(n);
    for (int r = 0; r < n; r++) fpos[olo[r]] = r;
    for (int r = 0; r < n; r++) f2b[r] = fpos[oup[r]];
    I.fwd2bwd.upload(f2b, s);
    HIPCHECK(hipStreamSynchronize(s));
  }
  HIPCHECK(hipStreamSynchronize(s));
  I.ready = true;
}

// ---------------------------------------------------------------------------------------
// factor / apply

template <class VT> static DBuf<VT>& LUbuf(Ilu& I);
template <> DBuf<double>& LUbuf<double>(Ilu& I) { return I.LU64; }
template <> DBuf<float>& LUbuf<float>(Ilu& I) { return I.LU32; }
template <class VT> static DBuf<VT>& PLbuf(Ilu& I);
template <> DBuf<double>& PLbuf<double>(Ilu& I) { return I.plo64; }
template <> DBuf<float>& PLbuf<float>(Ilu& I) { return I.plo32; }
template <class VT> static DBuf<VT>& PUbuf(Ilu& I);
template <> DBuf<double>& PUbuf<double>(Ilu& I) { return I.pup64; }
template <> DBuf<float>& PUbuf<float>(Ilu& I) { return I.pup32; }
// block sweep values of one precision: entries (lower, upper), unit couplings (lower, upper)
template <class VT> struct BSvals {
  DBuf<VT> *vlo, *vup, *wlo, *wup;
  DBuf<double>* rdg;
};
template <class VT> static BSvals<VT> bsvals(BlockSweep& B);
template <> BSvals<double> bsvals<double>(BlockSweep& B)
{
  return { &B.vlo64, &B.vup64, &B.wlo64, &B.wup64, &B.rdg64 };
}
template <> BSvals<float> bsvals<float>(BlockSweep& B)
{
  return { &B.vlo32, &B.vup32, &B.wlo32, &B.wup32, &B.rdg32 };
}
// chunk sweep values of one precision: entries, inverses (lower, upper)
template <class VT> struct CSvals {
  DBuf<VT> *vlo, *vup;
  DBuf<double> *tlo, *tup, *dgu;
};
template <class VT> static CSvals<VT> csvals(ChunkSweep& S);
template <> CSvals<double> csvals<double>(ChunkSweep& S)
{
  return { &S.vlo64, &S.vup64, &S.tlo64, &S.tup64, &S.dgu64 };
}
template <> CSvals<float> csvals<float>(ChunkSweep& S)
{
  return { &S.vlo32, &S.vup32, &S.tlo32, &S.tup32, &S.dgu32 };
}
// node sweep values of one precision: entries, couplings, reciprocal diagonals (upper)
template <class VT> struct NSvals {
  DBuf<VT> *v, *w;
  DBuf<double>* rdg;
};
template <class VT> static NSvals<VT> nsvals(NodeSweep& S);
template <> NSvals<double> nsvals<double>(NodeSweep& S) { return { &S.v64, &S.w64, &S.rdg64 }; }
template <> NSvals<float> nsvals<float>(NodeSweep& S) { return { &S.v32, &S.w32, &S.rdg32 }; }
template <class VT> static DBuf<VT>& PDbuf(Ilu& I);
template <> DBuf<double>& PDbuf<double>(Ilu& I) { return I.pdg64; }
template <> DBuf<float>& PDbuf<float>(Ilu& I) { return I.pdg32; }

template <class VT> static DBuf<VT>& FUbuf(Ilu& I);
template <> DBuf<double>& FUbuf<double>(Ilu& I) { return I.fu.u64; }
template <> DBuf<float>& FUbuf<float>(Ilu& I) { return I.fu.u32; }

template <class VT>
static void factor_t(Ctx& c, Ilu& I, const VT* A)
{
  DBuf<VT>& LU = LUbuf<VT>(I);
  LU.alloc(I.nnz);
  HIPCHECK(hipMemcpyAsync(LU.p, A, sizeof(VT) * I.nnz, hipMemcpyDeviceToDevice, c.stream));
  int* err = reinterpret_cast<int*>(c.red.p + 8);
  HIPCHECK(hipMemsetAsync(err, 0, sizeof(int), c.stream));
  auto need_rows = [&]() {
    if (I.fdesc.p) return;
    std::vector<int> scol(I.nnz);
    I.srt_cols.download(scol.data(), I.nnz, c.stream);
    HIPCHECK(hipStreamSynchronize(c.stream));
    build_rows(I, scol, c.stream);
  };
  const char* lv = getenv("RMX_ILU_LEVELS");
  if (!(lv && atoi(lv) == 1)) {
    if (!I.fu.sch) need_rows();
    // one persistent launch: rows in level order, pivot rows awaited by completion flags
    if (I.done.n != (size_t)I.n) {
      I.done.alloc(I.n);
      HIPCHECK(hipMemsetAsync(I.done.p, 0, sizeof(int) * I.n, c.stream));
      I.epoch = 0;
    }
    I.flow_state.alloc(4);
    if (++I.epoch == INT_MAX) {                   // epochs exhausted: clear the flags
      HIPCHECK(hipMemsetAsync(I.done.p, 0, sizeof(int) * I.n, c.stream));
      I.epoch = 1;
    }
    // one-wave workgroups, three per CU: enough rows in flight that a row is taken before
    // its pivot rows finish (about three levels ahead on the 2M-triangle meander), while
    // more waves lengthen every row (FP32 factorisation there: 640 waves 178 ms, 768
    // 168 ms, 896 182 ms, 1024 245 ms)
    hipDeviceProp_t prop;
    HIPCHECK(hipGetDeviceProperties(&prop, c.device));
    int per_cu = 0;
    HIPCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)k_ilu_flow<VT>,
                                                          64, 0));
    per_cu = std::max(1, std::min(per_cu, 3));
    int nwg = (int)std::min<long long>(I.n, (long long)per_cu * prop.multiProcessorCount);
    if (const char* e = getenv("RMX_ILU_WAVES")) nwg = std::max(1, std::min(nwg, atoi(e)));
    // by units three waves on two CUs: a wave that waits polls, and the polls slow the others'
    // loads (FP32, ms at 200 x 20, 80 x 320, 640 x 320 cells: 192 waves 1.2, 6.5, 25; 384 1.3,
    // 6.4, 17; 768 1.5, 7.8, 26; with the row-by-row kernel's pause between polls 384 waves
    // take 1.4, 7.4, 19)
    int nwu = 3 * prop.multiProcessorCount / 2;
    if (const char* e = getenv("RMX_ILU_WAVES")) nwu = std::max(1, std::min(4096, atoi(e)));
    int spin = 1 << 22;
    if (const char* e = getenv("RMX_ILU_SPIN")) spin = std::max(32, atoi(e));
    // a pass factors every row after skip; a pivot below 1e-20 is repaired as the
    // reference does (k_ilu_repair, on the first such row: every row before it is final),
    // and the rows after it are factored again from A
    int skip = -1;
    I.repaired = 0;
    for (;;) {
      int st[4] = {0, 0, 0, INT_MAX};
      HIPCHECK(hipMemcpyAsync(I.flow_state.p, st, sizeof(int) * 4, hipMemcpyHostToDevice,
                              c.stream));
      const int kt = kt_begin(c, KT_FACTOR, 3.0 * (double)I.nnz * (sizeof(VT) + 4));
      if (I.fu.sch && skip < 0) {
        const FlowSchedule& F = *I.fu.sch;
        DBuf<VT>& U = FUbuf<VT>(I);
        U.alloc(FU * (size_t)F.cols);
        k_unit_flow<VT><<<std::min(F.nu, nwu), 64, 0, c.stream>>>(
            F.desc.p, F.nu, F.list.p, F.plan.p, I.srt_pos.p, LU.p, U.p, I.done.p,
            I.epoch, I.flow_state.p, spin);
      } else {
        k_ilu_flow<VT><<<nwg, 64, 0, c.stream>>>(I.fdesc.p, I.n, I.cols.p, I.srt_cols.p,
                                                 I.srt_pos.p, I.fpiv.p, I.fpbase.p, I.plan.p,
                                                 LU.p, I.done.p, I.epoch, I.flow_state.p, spin,
                                                 skip);
      }
      kt_end(c, kt);
      HIPCHECK(hipGetLastError());
      HIPCHECK(hipMemcpyAsync(st, I.flow_state.p, sizeof(int) * 4, hipMemcpyDeviceToHost,
                              c.stream));
      HIPCHECK(hipStreamSynchronize(c.stream));
      if (st[FLOW_ABORT])
        fail(RMX_ERR_HIP, "ILU(0): a row's wait for its pivot rows exceeded its bound (dataflow "
                          "factorisation aborted)");
      if (!st[FLOW_ERR]) break;
      const int bad = st[FLOW_BADROW];
      if (bad <= skip || bad >= I.n) fail(RMX_ERR_HIP, "ILU(0): inconsistent pivot record");
      k_ilu_repair<VT><<<1, 64, 0, c.stream>>>(bad, I.rp.p, I.cols.p, I.srt_cols.p, I.srt_pos.p,
                                               A, LU.p, I.flow_state.p);
      HIPCHECK(hipGetLastError());
      HIPCHECK(hipMemcpyAsync(st, I.flow_state.p, sizeof(int) * 4, hipMemcpyDeviceToHost,
                              c.stream));
      HIPCHECK(hipStreamSynchronize(c.stream));
      if (st[FLOW_ERR] == 2)
        fail(RMX_ERR_PIVOT, "ILU(0) cannot be applied to the matrix: pivot of row " +
                            std::to_string(bad) + " below 1e-20 and no later row of its pattern "
                            "holds its column (PRECO_ILU0::Factor - 1)");
      I.repaired++;
      // the rows after it: the matrix again, not finished
      const long long q1 = I.h_rp[bad + 1];
      if (I.nnz > q1)
        HIPCHECK(hipMemcpyAsync(LU.p + q1, A + q1, sizeof(VT) * (I.nnz - q1),
                                hipMemcpyDeviceToDevice, c.stream));
      if (bad + 1 < I.n)
        k_flags_clear<<<(I.n - bad - 1 + 255) / 256, 256, 0, c.stream>>>(bad + 1, I.n, I.done.p);
      HIPCHECK(hipGetLastError());
      skip = bad;
      need_rows();
    }
  } else {
  need_rows();
  const long long plan_n = (long long)I.plan.n;
  const int kt = kt_begin(c, KT_FACTOR, 3.0 * (double)I.nnz * (sizeof(VT) + 4));
  for (size_t l = 0; l + 1 < I.flev.size(); l++) {
    const int a = I.flev[l], cnt = I.flev[l + 1] - a;
    const bool last = l + 2 >= I.flev.size();
    const int an = last ? a : I.flev[l + 1];
    const int cntn = last ? 0 : I.flev[l + 2] - an;
    k_ilu_level<VT><<<cnt, 64, 0, c.stream>>>(I.fdesc.p + a, cnt, I.cols.p, I.srt_cols.p,
                                              I.srt_pos.p, I.fpiv.p, I.fpbase.p + a,
                                              I.plan.p, LU.p, err,
                                              I.fdesc.p + an, cntn, I.fpbase.p + an, plan_n);
  }
  kt_end(c, kt);
  }
  HIPCHECK(hipGetLastError());
  if (I.lo.packed) {                            // level sweeps
    DBuf<VT>& pl = PLbuf<VT>(I);
    DBuf<VT>& pu = PUbuf<VT>(I);
    DBuf<VT>& pd = PDbuf<VT>(I);
    pl.alloc(std::max<long long>(I.lo.ne, 1));
    pu.alloc(std::max<long long>(I.up.ne, 1));
    pd.alloc(I.n);
    if (I.lo.ne) k_pack<VT><<<4096, 256, 0, c.stream>>>(I.lo.ne, I.lo.psrc.p, LU.p, pl.p);
    if (I.up.ne) k_pack<VT><<<4096, 256, 0, c.stream>>>(I.up.ne, I.up.psrc.p, LU.p, pu.p);
    k_pack_diag<VT><<<(I.n + 255) / 256, 256, 0, c.stream>>>(I.n, I.up.prow.p, I.rp.p, LU.p, pd.p);
  }
  if (I.nlo.on && I.nup.on) {                   // node sweeps
    for (NodeSweep* S : { &I.nlo, &I.nup }) {
      const NSvals<VT> V = nsvals<VT>(*S);
      V.v->alloc(S->src.n);
      V.w->alloc(S->wsrc.n);
      k_pack<VT><<<4096, 256, 0, c.stream>>>((long long)S->src.n, S->src.p, LU.p, V.v->p);
      k_pack<VT><<<1024, 256, 0, c.stream>>>((long long)S->wsrc.n, S->wsrc.p, LU.p, V.w->p);
    }
    DBuf<double>& rd = *nsvals<VT>(I.nup).rdg;
    rd.alloc(I.n);
    k_rcp_diag<VT><<<(I.n + 255) / 256, 256, 0, c.stream>>>(I.n, I.rp.p, LU.p, rd.p);
  }
  if (I.cs.on) {                                // chunk sweeps: values, inverses
    ChunkSweep& S = I.cs;
    const CSvals<VT> V = csvals<VT>(S);
    V.vlo->alloc(S.slo.n);
    V.vup->alloc(S.sup.n);
    V.tlo->alloc((size_t)(S.nch + CH_DEEP2) * CH_T);      // loads ahead end past the last chunk
    V.tup->alloc((size_t)(S.nch + CH_DEEP2) * CH_T);
    V.dgu->alloc((size_t)(S.nch + CH_DEEP2) * CH_ROWS);
    k_pack<VT><<<4096, 256, 0, c.stream>>>((long long)S.slo.n, S.slo.p, LU.p, V.vlo->p);
    k_pack<VT><<<4096, 256, 0, c.stream>>>((long long)S.sup.n, S.sup.p, LU.p, V.vup->p);
    k_chunk_inv<VT><<<S.nch, 64, 0, c.stream>>>(S.chunks.p, S.rows.p, S.slot.p, I.rp.p, I.cols.p,
                                                LU.p, V.tlo->p, V.tup->p, V.dgu->p);
  }
  if (I.bs.on) {                                // block sweeps: values in their entry order
    BlockSweep& B = I.bs;
    const BSvals<VT> V = bsvals<VT>(B);
    const std::pair<DBuf<VT>*, const DBuf<int>*> packs[4] = {
      { V.vlo, &B.slo }, { V.vup, &B.sup }, { V.wlo, &B.sulo }, { V.wup, &B.suup } };
    for (const auto& pk : packs) {
      pk.first->alloc(pk.second->n);
      k_pack<VT><<<4096, 256, 0, c.stream>>>((long long)pk.second->n, pk.second->p, LU.p,
                                             pk.first->p);
    }
    V.rdg->alloc(B.sdg.n);
    k_pack_rcp<VT><<<4096, 256, 0, c.stream>>>((long long)B.sdg.n, B.sdg.p, LU.p, V.rdg->p);
  }
  HIPCHECK(hipGetLastError());
  int h_err = 0;
  HIPCHECK(hipMemcpyAsync(&h_err, err, sizeof(int), hipMemcpyDeviceToHost, c.stream));
  HIPCHECK(hipStreamSynchronize(c.stream));
  if (h_err)
    fail(RMX_ERR_PIVOT, "ILU(0): pivot below 1e-20 (the per-level factorisation, "
                        "RMX_ILU_LEVELS=1, does not repair pivots; the dataflow one does)");
}

void ilu_factor(Ctx& c, Ilu& I, int prec)
{
  if (!I.ready) fail(RMX_ERR_ARG, "ILU(0): no schedule");
  if (prec == RMX_F32) {
    if (!c.have32) fail(RMX_ERR_ARG, "ILU(0) FP32: no FP32 matrix (assemble or convert first)");
    factor_t<float>(c, I, c.A32.p);
    I.fac32 = true;
  } else {
    if (!c.have64) fail(RMX_ERR_ARG, "ILU(0) FP64: no FP64 matrix");
    factor_t<double>(c, I, c.A64.p);
    I.fac64 = true;
  }
}

template <class VT>
static void launch_sweeps(Ctx& c, Ilu& I, const double* b, double* x, hipEvent_t* ev,
                          const int* aidx, const double* aval)
{
  // 4 lanes per row with 12 / 6 register entries each, 512 threads (two workgroups per compute
  // unit by registers and LDS)
  const int nb = I.nblk;
  const int nt = STAGE_THREADS;
  if (ev) HIPCHECK(hipEventRecord(ev[0], c.stream));
  const double vb = (double)sizeof(VT) + 4.0;
  int kt = kt_begin(c, KT_SWEEP_LO, (double)I.lo.ne * vb + 20.0 * I.n);
  k_sweep_stage<VT, true, 4, 12><<<nb, nt, 0, c.stream>>>(I.lo.blev.p, I.lo.bpos.p,
      I.lo.lev_ptr.p, I.lo.prs.p, I.lo.pcol.p, PLbuf<VT>(I).p, nullptr, I.lo.prow.p, b, nullptr,
      nullptr, I.lo.xp.p, nullptr, nullptr);
  kt_end(c, kt);
  if (ev) HIPCHECK(hipEventRecord(ev[1], c.stream));
  kt = kt_begin(c, KT_SWEEP_UP, (double)I.up.ne * vb + 24.0 * I.n);
  k_sweep_stage<VT, false, 4, 6><<<nb, nt, 0, c.stream>>>(I.up.blev.p, I.up.bpos.p,
      I.up.lev_ptr.p, I.up.prs.p, I.up.pcol.p, PUbuf<VT>(I).p, PDbuf<VT>(I).p, I.fwd2bwd.p,
      I.lo.xp.p, I.up.prow.p, x, I.up.xp.p, aidx, aval);
  kt_end(c, kt);
  if (ev) HIPCHECK(hipEventRecord(ev[2], c.stream));
  HIPCHECK(hipGetLastError());
}

// Both sweeps of every block in one launch (one wave per block).
template <class VT>
static void launch_blocks(Ctx& c, Ilu& I, const double* b, double* x, hipEvent_t* ev,
                          const int* aidx, const double* aval)
{
  BlockSweep& B = I.bs;
  const BSvals<VT> V = bsvals<VT>(B);
  if (ev) HIPCHECK(hipEventRecord(ev[0], c.stream));
  // algorithmic bytes: entry values, a 2-byte column per node and column, per node 16 coupling
  // values and 4 FP64 reciprocal diagonals (those of 3 rows used), per row the gather index, right-hand
  // side and result, per slot its descriptor, per pass its table entry, the folded prolongation
  const double v = (double)sizeof(VT);
  const double bytes = (double)(B.ne_lo + B.ne_up) * v + 2.0 * B.ncol + (double)B.nunit * (32.0 + 16.0 * v) +
                       8.0 * B.nslot + 20.0 * I.n + 4.0 * B.npass + (aidx ? 12.0 * I.n : 0.0);
  const int kt = kt_begin(c, KT_SWEEP_BLK, bytes);
  k_block_sweep<VT><<<B.nb, 64, B.lds, c.stream>>>(B.info.p, B.gidx.p, B.tab.p, B.desc.p,
      V.vlo->p, reinterpret_cast<const uint2*>(B.clo.p), V.wlo->p, V.vup->p,
      reinterpret_cast<const uint2*>(B.cup.p), V.wup->p, V.rdg->p, b, x, aidx, aval);
  kt_end(c, kt);
  if (ev) {
    HIPCHECK(hipEventRecord(ev[1], c.stream));
    HIPCHECK(hipEventRecord(ev[2], c.stream));
  }
  HIPCHECK(hipGetLastError());
}

template <class VT>
static void launch_chunks(Ctx& c, Ilu& I, const double* b, double* x, hipEvent_t* ev,
                          const int* aidx, const double* aval)
{
  ChunkSweep& S = I.cs;
  const CSvals<VT> V = csvals<VT>(S);
  if (ev) HIPCHECK(hipEventRecord(ev[0], c.stream));
  // algorithmic bytes: entry values and 2-byte columns, the inverses of the chunks, per row the
  // gather index twice, right-hand side and result, the folded prolongation
  const double bytes = (double)S.ne * (sizeof(VT) + 2.0) + 16.0 * CH_T * S.nch +
                       32.0 * I.n + (aidx ? 12.0 * I.n : 0.0);
  const int kt = kt_begin(c, KT_SWEEP_BLK, bytes);
  auto run = [&](auto* kernel) {
    kernel<<<S.nb, 64, S.lds, c.stream>>>(S.info.p, S.rows.p, S.dlo.p, S.ilo.p, V.vlo->p, V.tlo->p,
                                          S.dup.p, S.iup.p, V.vup->p, V.tup->p, V.dgu->p, b, x, aidx, aval);
  };
  if (S.ahead == 2) run(k_chunk_sweep<VT, 2>);
  else run(k_chunk_sweep<VT, CH_PK>);
  kt_end(c, kt);
  if (ev) {
    HIPCHECK(hipEventRecord(ev[1], c.stream));
    HIPCHECK(hipEventRecord(ev[2], c.stream));
  }
  HIPCHECK(hipGetLastError());
}

template <class VT, bool LOWER>
static void launch_nodes(Ctx& c, Ilu& I, NodeSweep& S, const double* b, double* x)
{
  const NSvals<VT> V = nsvals<VT>(S);
  auto run = [&](auto* kernel) {
    if (S.lds > 65536)
      HIPCHECK(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   NS_LDS));
    kernel<<<I.nblk, 64 * S.waves, S.lds, c.stream>>>(S.info.p, S.tab.p, S.desc.p, V.v->p,
        reinterpret_cast<const uint2*>(S.cols.p), V.w->p, V.rdg->p, b, x);
  };
  const SweepSet& L = LOWER ? I.lo : I.up;
  const int kt = kt_begin(c, LOWER ? KT_SWEEP_LO : KT_SWEEP_UP,
                          (double)L.ne * (sizeof(VT) + 4.0) + (LOWER ? 20.0 : 24.0) * I.n);
  if (S.lgmax == 0) run(k_node_sweep<VT, LOWER, 0>);
  else if (S.lgmax == 1) run(k_node_sweep<VT, LOWER, 1>);
  else run(k_node_sweep<VT, LOWER, 2>);
  kt_end(c, kt);
}

// The sweeps that an application runs (RMX_SWEEPS_*).
int ilu_sweeps(const Ilu& I)
{
  if (sweep_variant() < 2 && I.lo.packed) return RMX_SWEEPS_LEVELS;
  if (I.cs.on) return RMX_SWEEPS_CHUNKS;
  if (I.bs.on) return RMX_SWEEPS_BLOCKS;
  return I.nlo.on && I.nup.on ? RMX_SWEEPS_NODES : RMX_SWEEPS_LEVELS;
}

template <class VT>
static bool apply_t(Ctx& c, Ilu& I, const double* b, double* x, hipEvent_t* ev, const int* aidx,
                    const double* aval)
{
  const int sw = ilu_sweeps(I);
  if (sw == RMX_SWEEPS_CHUNKS) { launch_chunks<VT>(c, I, b, x, ev, aidx, aval); return aidx != nullptr; }
  if (sw == RMX_SWEEPS_BLOCKS) { launch_blocks<VT>(c, I, b, x, ev, aidx, aval); return aidx != nullptr; }
  if (sw == RMX_SWEEPS_NODES) {
    if (ev) HIPCHECK(hipEventRecord(ev[0], c.stream));
    launch_nodes<VT, true>(c, I, I.nlo, b, I.lo.xp.p);
    if (ev) HIPCHECK(hipEventRecord(ev[1], c.stream));
    launch_nodes<VT, false>(c, I, I.nup, I.lo.xp.p, x);
    if (ev) HIPCHECK(hipEventRecord(ev[2], c.stream));
    HIPCHECK(hipGetLastError());
    return false;
  }
  launch_sweeps<VT>(c, I, b, x, ev, aidx, aval);
  return aidx != nullptr;
}

bool ilu_apply(Ctx& c, Ilu& I, int prec, const double* b, double* x, hipEvent_t* ev,
               const int* aidx, const double* aval)
{
  if (prec == RMX_F32) {
    if (!I.fac32) fail(RMX_ERR_ARG, "ILU(0) FP32 not factored");
    return apply_t<float>(c, I, b, x, ev, aidx, aval);
  }
  if (!I.fac64) fail(RMX_ERR_ARG, "ILU(0) FP64 not factored");
  return apply_t<double>(c, I, b, x, ev, aidx, aval);
}

// ---- the context's two instances ----

// Segments per strip: the requested count, or blocks of about 560 rows (at most 32 per
// strip).  Blocks much smaller than that drop most of the factor's couplings from the
// sweeps: on a 23k-equation meander reach, 32 segments of its 11 strips (66-row blocks)
// left FGMRES stalled where blocks of ~700 rows converge.
static int strip_segments(const Ctx& c, int nblk)
{
  if (c.segments > 0) return c.segments;
  const long long rows = c.n / std::max(1, nblk);
  return (int)std::max<long long>(1, std::min<long long>(32, rows / 560));
}

void setup_ilu_schedule(Ctx& c)
{
  std::vector<int> hrp, hcols;
  if (c.csr_only) {
    hrp.resize(c.n + 1); hcols.resize(c.nnz);
    c.rowptr.download(hrp.data(), c.n + 1, c.stream);
    c.cols.download(hcols.data(), c.nnz, c.stream);
    HIPCHECK(hipStreamSynchronize(c.stream));
  }
  const std::vector<int>& rp = c.csr_only ? hrp : c.hm.rowptr;
  const std::vector<int>& cl = c.csr_only ? hcols : c.hm.cols;
  std::vector<int> group, unit(c.n);
  if (!c.csr_only) {
    group.assign(c.n, -1);
    for (size_t k = 0; k < c.hm.eqno.size(); k++)
      if (c.hm.eqno[k] >= 0) group[c.hm.eqno[k]] = (int)(k / 3);
    unit = group;
  } else {
    // rows that follow each other with one set of columns, as the rows of a node have it
    std::vector<char> mark(c.n, 0);
    for (int i = 0; i < c.n; i++) {
      bool same = i > 0 && rp[i + 1] - rp[i] == rp[i] - rp[i - 1];
      if (same) {
        for (int q = rp[i - 1]; q < rp[i]; q++) mark[cl[q]] = 1;
        for (int q = rp[i]; q < rp[i + 1]; q++) same = same && mark[cl[q]];
        for (int q = rp[i - 1]; q < rp[i]; q++) mark[cl[q]] = 0;
      }
      unit[i] = same ? unit[i - 1] : i;
    }
  }
  std::vector<int> scol;
  std::vector<unsigned char> spos;
  const bool twice = sorted_columns(rp, cl, scol, spos);
  ilu_setup(c.ilu, c.n, rp, cl, 1, nullptr, unit, c.stream, nullptr, 1, 0, scol, spos, nullptr, twice);
  // strip ILU: two strips per compute unit (two sweep workgroups fit one CU's LDS), at
  // least a few thousand rows each
  hipDeviceProp_t prop;
  HIPCHECK(hipGetDeviceProperties(&prop, c.device));
  int nblk = c.strips > 0 ? c.strips : 2 * prop.multiProcessorCount;
  nblk = std::max(1, std::min(nblk, c.n / 2048));
  ilu_setup(c.silu, c.n, rp, cl, nblk, c.csr_only ? nullptr : &group, unit, c.stream,
            c.csr_only ? nullptr : &c.hm, strip_segments(c, nblk), STAGE_ROWS, scol, spos, &c.ilu, twice);
  c.coarse.ready = c.coarse.fac = false;
  const int cseg = coarse_segments_of(c);
  if (!c.csr_only && cseg > 0) coarse_setup(c, rp, cl, group, cseg);
}

Ilu& ilu_of(Ctx& c, int kind)
{
  return (kind == RMX_PREC_SILU0 || kind == RMX_PREC_SILU0C || kind == RMX_PREC_MPNN) ? c.silu : c.ilu;
}

void dev_ilu0_factor(Ctx& c, int prec) { ilu_factor(c, c.ilu, prec); }

void dev_ilu0_apply(Ctx& c, int prec, const double* b, double* x)
{
  ilu_apply(c, c.ilu, prec, b, x, nullptr);
}

// Average kernel durations (HIP events on the context stream) of SpMV and of the two
// sweeps of an ILU instance, `reps` times each on the current system.
void dev_profile(Ctx& c, int prec, int reps, rmx_kernel_times& out)
{
  hipEvent_t ev[3];
  for (auto& e : ev) HIPCHECK(hipEventCreate(&e));
  double* xv = c.w[0].p;
  double* yv = c.w[1].p;
  double t_spmv = 0, t_fwd = 0, t_bwd = 0, t_sf = 0, t_sb = 0;
  dev_spmv(c, prec, c.B.p, yv);         // untimed: brings a re-laid-out matrix up to date
  for (int r = 0; r < reps; r++) {
    HIPCHECK(hipEventRecord(ev[0], c.stream));
    dev_spmv(c, prec, c.B.p, yv);
    HIPCHECK(hipEventRecord(ev[1], c.stream));
    HIPCHECK(hipEventSynchronize(ev[1]));
    float ms = 0;
    HIPCHECK(hipEventElapsedTime(&ms, ev[0], ev[1]));
    t_spmv += ms * 1e-3;
    for (int k = 0; k < 2; k++) {
      Ilu& I = k == 0 ? c.ilu : c.silu;
      if (!((prec == RMX_F32) ? I.fac32 : I.fac64)) continue;
      ilu_apply(c, I, prec, c.B.p, xv, ev);
      HIPCHECK(hipEventSynchronize(ev[2]));
      float m1 = 0, m2 = 0;
      HIPCHECK(hipEventElapsedTime(&m1, ev[0], ev[1]));
      HIPCHECK(hipEventElapsedTime(&m2, ev[1], ev[2]));
      if (k == 0) { t_fwd += m1 * 1e-3; t_bwd += m2 * 1e-3; }
      else { t_sf += m1 * 1e-3; t_sb += m2 * 1e-3; }
    }
  }
  for (auto& e : ev) HIPCHECK(hipEventDestroy(e));
  out.spmv_s = t_spmv / reps;
  out.ilu_fwd_s = t_fwd / reps;
  out.ilu_bwd_s = t_bwd / reps;
  out.ilu_apply_s = out.ilu_fwd_s + out.ilu_bwd_s;
  out.silu_fwd_s = t_sf / reps;
  out.silu_bwd_s = t_sb / reps;
  out.n_spmv = reps;
  out.n_ilu = reps;
  out.spmv_bytes = prec == RMX_F32 ? spmv_f32_bytes(c)
                                   : (double)c.nnz * 12.0 + 4.0 * (c.n + 1) + 16.0 * c.n;
}

}  // namespace rmx
