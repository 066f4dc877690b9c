// Forward combine: out[idx[g], :] += w[g] * X_e[g - off[e], :]
//
// Replaces _launch_grouped_kernel + _grouped_weighted_scatter_add_kernel
// (src/fastmoe/kernels/ops.py:277-310, :57-194).  Three modes:
//
// DET (token-major).  A wave owns one (token, column chunk).  It walks the token's plan segment in
// ascending packed-row order (ordering a short segment in registers first), loads 16 bytes per
// lane per row straight from each expert's buffer
// (the record carries the row address), multiplies by the gate in fp32, adds into fp32 registers
// and writes the output chunk once.  Every output byte is written exactly once and every expert
// byte read exactly once, so HBM traffic equals the compulsory bytes; no zero-fill is needed and
// the result is bit-identical run to run (and, in fp32, to the CPU index_add_ path, which adds the
// rounded products in the same ascending order).
//
// ATOMIC (packed-row-major, the reference kernel's order).  A wave owns one (row g, column chunk):
// binary-searches g's expert in the offsets (ops.py:151-154 does offsets + program id instead),
// loads the row, scales it and adds it into out[idx[g]] with global_atomic_add_f32.  A 16-bit
// output is accumulated in an fp32 workspace (initialised from out, or zeroed) and converted once
// at the end, so it is the fp32 sum rounded once, like the deterministic mode's; only the order of
// the fp32 additions differs run to run.
//
// ATOMIC_PACKED.  As ATOMIC, but a 16-bit output takes gfx950's packed atomics
// (global_atomic_pk_add_bf16 / _f16) on element pairs directly: no workspace and half the atomic
// requests, but every add rounds to 16 bits (the reference kernel's behaviour with a bf16 output).
#include <algorithm>

#include "plan.h"

namespace fmoe {

// acc += w[i] * row i, for the cnt records of a batch held one per lane, in record order: R rows of
// U vectors per lane in flight.  The spare slots of a partial batch load through an empty range
// (num_records 0): the hardware range check returns zeros without a memory request, so every load
// is issued unconditionally and none is wasted.
template <typename TX, int V, int U, int R, bool AL>
__device__ __forceinline__ void add_rows(const LaneRecs& lr, int cnt, uint32_t xrow_bytes,
                                         const uint32_t (&xoff)[U], float (&acc)[U][V]) {
  using VX = Vec<TX, V>;
  for (int i = 0; i < cnt; i += R) {
    typename VX::raw_t a[R][U];
    float wr[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int ir = min(i + r, cnt - 1);
      const rsrc_t rx = make_rsrc(lr.src(ir), i + r < cnt ? xrow_bytes : 0u);
      wr[r] = lr.w(ir);
#pragma unroll
      for (int u = 0; u < U; ++u) a[r][u] = load_x<TX, V, AL>(rx, xoff[u]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      // Used whether or not the row exists, so that the compiler does not move the row's loads
      // into the branch below, behind the other rows'.
#pragma unroll
      for (int u = 0; u < U; ++u) asm volatile("" : "+v"(a[r][u]));
      if (i + r < cnt) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          float x[V];
          VX::cvt(a[r][u], x);
#pragma unroll
          for (int v = 0; v < V; ++v) acc[u][v] = acc[u][v] + x[v] * wr[r];
        }
      }
    }
  }
}

// Tile of one wave unit: U 16-byte vectors per lane per row (64 * V * U columns) and batches of
// R rows, so R * U independent loads per lane are in flight before the first use.
template <typename TX, typename TO, int V, int U, int RB, bool AL>
__device__ __forceinline__ void fwd_det_body(const int32_t* __restrict__ row_ptr,
                                             const Rec* __restrict__ rec, TO* __restrict__ out,
                                             int64_t out_stride, uint32_t D, uint32_t t,
                                             uint32_t chunk, int accumulate, int out_stream) {
  using VO = Vec<TO, V>;
  constexpr int CW = kWave * V * U;
  // The misaligned-row path (element loads) takes one row at a time so that it does not set the
  // register budget of the kernel.
  constexpr int R = AL ? RB : 1;
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t col0 = chunk * CW + (uint32_t)lane * V;
  uint32_t xoff[U], ooff[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    xoff[u] = (col0 + (uint32_t)u * kWave * V) * (uint32_t)sizeof(TX);
    ooff[u] = (col0 + (uint32_t)u * kWave * V) * (uint32_t)sizeof(TO);
  }
  const uint32_t xrow_bytes = D * (uint32_t)sizeof(TX);
  const int beg = row_ptr[t];
  const int end = row_ptr[t + 1];
  const rsrc_t ro = make_rsrc(out + (int64_t)t * out_stride, D * (uint32_t)sizeof(TO));

  float acc[U][V];
  if (accumulate) {
    if (beg == end) return;  // nothing routed here: out keeps its contents
#pragma unroll
    for (int u = 0; u < U; ++u) VO::cvt(VO::ld(ro, ooff[u]), acc[u]);
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int v = 0; v < V; ++v) acc[u][v] = 0.f;
  }

  for (int jb = beg; jb < end; jb += kWave) {
    const int cnt = min(end - jb, kWave);
    LaneRecs lr;
    lr.load(rec, jb, cnt, lane);
    // A segment of up to 64 rows comes unordered from the plan: order it by g here.  Longer
    // segments are already in ascending g.
    if (end - beg <= kWave) lr.sort_by_row(cnt, lane);
    add_rows<TX, V, U, R, AL>(lr, cnt, xrow_bytes, xoff, acc);
  }
  // columns >= D: dropped by range check
  if (out_stream) {  // wave-uniform
#pragma unroll
    for (int u = 0; u < U; ++u) VO::template st<kCPol>(ro, ooff[u], acc[u]);
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) VO::template st<FMOE_OUT_CPOL>(ro, ooff[u], acc[u]);
  }
}

template <typename TX, typename TO, int V, int U, int RB>
__global__ __launch_bounds__(kGroup) void k_fwd_det(const int32_t* __restrict__ status,
                                                    const int32_t* __restrict__ row_ptr,
                                                    const Rec* __restrict__ rec,
                                                    TO* __restrict__ out, int64_t out_stride,
                                                    uint32_t D, uint32_t T, uint32_t chunks,
                                                    int accumulate, int out_stream) {
  const bool al = !(V > 1 && status[kStatusMisaligned] != 0);
  const uint32_t units = T * chunks;
  // Wave units (token, column chunk); a grid smaller than units / 4 strides over them.
  for (uint32_t unit = blockIdx.x * kWavesPerGroup + (uint32_t)uniform(threadIdx.x / kWave);
       unit < units; unit += gridDim.x * kWavesPerGroup) {
    const uint32_t t = unit / chunks;
    const uint32_t chunk = unit - t * chunks;
    if (al)
      fwd_det_body<TX, TO, V, U, RB, true>(row_ptr, rec, out, out_stride, D, t, chunk, accumulate,
                                           out_stream);
    else
      fwd_det_body<TX, TO, V, U, RB, false>(row_ptr, rec, out, out_stride, D, t, chunk, accumulate,
                                            out_stream);
  }
}

// ---- backward of the dispatch permutation ------------------------------------------------------
// grad_x[t, :] = sum of the packed-row gradients of token t's k slots, in ascending packed-row
// order, and (GATES) grad_gates[i] = grad_sorted[slot_pos[i]].  The slot map is the token-major
// inverse already: slot t * k + j sits at packed row slot_pos[t * k + j] of one buffer, so a wave
// makes its records in registers from one load and the combine needs no plan, no unit gates and no
// launch but this one.  A wave owns a (token, column chunk) and sums with k_fwd_det's arithmetic
// (unit gates: x * 1), so the result is the planned combine's bit for bit; the wave of chunk 0
// moves the token's gate gradients.  A slot_pos entry outside [0, N) adds nothing.
// Bound by HBM like k_fwd_det.  T=8192, D=4096, top-6, bf16, permutation and its backward: 195.6 us
// with the slot-map plan, the combine and the gate-gradient kernel (and autograd's fills of the
// integer outputs' gradients), 184.4 us with this kernel alone and k_fwd_det's tiles of then.
template <typename TX, int V, int U, int RB, bool GATES, typename TG>
__global__ __launch_bounds__(kGroup) void k_slots_bwd(const int32_t* __restrict__ slot_pos,
                                                      uint32_t k, uint32_t N,
                                                      const TX* __restrict__ rows, uint32_t D,
                                                      uint32_t T, uint32_t chunks,
                                                      TX* __restrict__ out, int out_stream,
                                                      const TG* __restrict__ gates,
                                                      TG* __restrict__ grad_gates) {
  using VX = Vec<TX, V>;
  constexpr int CW = kWave * V * U;
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t unit = blockIdx.x * kWavesPerGroup + (uint32_t)uniform(threadIdx.x / kWave);
  const uint32_t t = unit / chunks;
  if (t >= T) return;  // wave-uniform
  const uint32_t chunk = unit - t * chunks;
  const uint32_t row_bytes = D * (uint32_t)sizeof(TX);
  const uint32_t slot = t * k + (uint32_t)lane;
  const bool mine = (uint32_t)lane < k;
  const uint32_t pos = mine ? (uint32_t)slot_pos[slot] : N;
  const bool ok = pos < N;  // a negative entry is a large unsigned one
  if (GATES && chunk == 0 && mine) grad_gates[slot] = ok ? gates[pos] : TG{};
  LaneRecs lr;
  lr.g = ok ? (int32_t)pos : 0x7fffffff;  // entries out of range sort behind the others
  const uint64_t src = (uint64_t)(uintptr_t)rows + (uint64_t)(ok ? pos : 0u) * row_bytes;
  lr.src_lo = (uint32_t)src;
  lr.src_hi = (uint32_t)(src >> 32);
  lr.w_bits = __float_as_uint(1.f);
  const int cnt = __builtin_popcountll(__ballot(ok));
  lr.sort_by_row((int)k, lane);
  uint32_t off[U];
  float acc[U][V];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    off[u] = (chunk * CW + (uint32_t)lane * V + (uint32_t)u * kWave * V) * (uint32_t)sizeof(TX);
#pragma unroll
    for (int v = 0; v < V; ++v) acc[u][v] = 0.f;
  }
  add_rows<TX, V, U, RB, true>(lr, cnt, row_bytes, off, acc);
  const rsrc_t ro = make_rsrc(out + (int64_t)t * D, row_bytes);
  // columns >= D: dropped by range check
  if (out_stream) {  // wave-uniform
#pragma unroll
    for (int u = 0; u < U; ++u) VX::template st<kCPol>(ro, off[u], acc[u]);
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) VX::template st<FMOE_OUT_CPOL>(ro, off[u], acc[u]);
  }
}

// ---- small inputs: the deterministic forward without a plan --------------------------------
// For at most kSmallRows rows the plan is not worth its own launch.  Every workgroup stages the
// token id of each row in LDS (-1 for an index outside [0, T)); a wave owns one (token, column
// chunk) unit as in k_fwd_det and finds the token's rows by ballots over the staged ids in
// ascending row order, 256 ids per step (four per lane in one 16-byte LDS read), compacting them
// through a window and taking them 64 at a time.  With 64 ids per step the scan bound the kernel
// from about 1024 rows; the kernel in us (bf16, T, D, top-k; launches in a graph), plan + k_fwd_det
// beside it:  64, 7168, 8: 6.0 (11.5)   128, 7168, 8: 7.1 (14.2)   256, 7168, 8: 9.7 (14.6)
// 512, 7168, 8: 17.2 (18.1)   1024, 1024, 4: 10.0 (11.2)   4096, 2048, 1: 15.5 (13.8).
// Lanes look up their row's expert in an LDS copy of the argument table.  The rows are added in
// ascending g with k_fwd_det's arithmetic, so the result is the same, bit for bit.
static_assert(kMetaChunk == kGroup, "one expert per thread copies the argument table");
constexpr int kSmallIds = 4;                   // staged ids per lane per step: one 16-byte LDS read
constexpr int kSmallStep = kWave * kSmallIds;  // ids per step
static_assert(kSmallRows % kSmallStep == 0, "whole steps");
template <typename TX, typename TO, int V, int U, bool AL>
__global__ __launch_bounds__(kGroup) void k_fwd_small(const HostTable meta,
                                                      const void* __restrict__ idx, int idx_dtype,
                                                      const void* __restrict__ w, int w_dtype,
                                                      uint32_t N, uint32_t T, uint32_t D,
                                                      uint32_t chunks, TO* __restrict__ out,
                                                      int64_t out_stride, int accumulate,
                                                      int32_t* __restrict__ status) {
  using VO = Vec<TO, V>;
  constexpr int CW = kWave * V * U;
  constexpr int R = AL ? 4 : 1;  // rows per batch of loads (one at a time for element loads)
  __shared__ __attribute__((aligned(16))) uint32_t tok[kSmallRows];
  __shared__ int win[kWavesPerGroup][kWave + kSmallStep];
  __shared__ int off_lds[kMetaChunk + 1];
  __shared__ uint64_t ptr_lds[kMetaChunk];
  __shared__ int invalid;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = uniform(tid / kWave);
  if (tid == 0) invalid = 0;
  small_table_to_lds(meta, off_lds, ptr_lds);
  __syncthreads();
  int bad = 0;
  const uint32_t padded = (N + kSmallStep - 1) / kSmallStep * kSmallStep;
  for (uint32_t g = tid; g < padded; g += kGroup) {
    const int64_t v = g < N ? load_index(idx, idx_dtype, g) : -1;
    const bool ok = v >= 0 && v < (int64_t)T;
    tok[g] = ok ? (uint32_t)v : 0xffffffffu;
    bad += ok || g >= N ? 0 : 1;
  }
  if (blockIdx.x == 0 && bad) atomicAdd(&invalid, bad);
  __syncthreads();
  if (blockIdx.x == 0 && tid == 0) status[kStatusInvalid] = invalid;

  const uint32_t xrow_bytes = D * (uint32_t)sizeof(TX);
  const int ne = meta.count;
  const uint32_t units = T * chunks;
  for (uint32_t unit = blockIdx.x * kWavesPerGroup + (uint32_t)wave; unit < units;
       unit += gridDim.x * kWavesPerGroup) {
    const uint32_t t = unit / chunks;
    const uint32_t chunk = unit - t * chunks;
    const uint32_t col0 = chunk * CW + (uint32_t)lane * V;
    uint32_t xoff[U], ooff[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      xoff[u] = (col0 + (uint32_t)u * kWave * V) * (uint32_t)sizeof(TX);
      ooff[u] = (col0 + (uint32_t)u * kWave * V) * (uint32_t)sizeof(TO);
    }
    const rsrc_t ro = make_rsrc(out + (int64_t)t * out_stride, D * (uint32_t)sizeof(TO));
    float acc[U][V];
    if (accumulate) {
#pragma unroll
      for (int u = 0; u < U; ++u) VO::cvt(VO::ld(ro, ooff[u]), acc[u]);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int v = 0; v < V; ++v) acc[u][v] = 0.f;
    }
    int have = 0;  // rows in the window (wave-uniform)
    int seen = 0;
    for (uint32_t base = 0; base < padded; base += kSmallStep) {
      // a lane's kSmallIds consecutive ids, then the next lane's: ascending rows
      const u32x4 id = *reinterpret_cast<const u32x4*>(&tok[base + (uint32_t)lane * kSmallIds]);
      uint64_t m[kSmallIds];
      uint64_t any = 0;
#pragma unroll
      for (int r = 0; r < kSmallIds; ++r) {
        m[r] = __ballot(id[r] == t);
        any |= m[r];
      }
      const bool last = base + kSmallStep >= padded;
      if (any) {  // wave-uniform
        int at = have;
#pragma unroll
        for (int r = 0; r < kSmallIds; ++r) at += lanes_below(m[r]);
#pragma unroll
        for (int r = 0; r < kSmallIds; ++r) {
          if (id[r] == t) win[wave][at++] = (int)(base + (uint32_t)lane * kSmallIds + r);
          have += __builtin_popcountll(m[r]);
        }
      }
      int head = 0;
      while (have - head >= kWave || (last && have > head)) {
        const int cnt = min(have - head, kWave);
        LaneRecs lr;
        lr.g = lane < cnt ? win[wave][head + lane] : 0;
        if (lane < cnt) {
          const int e = expert_of_row32(off_lds, ne, lr.g);
          const uint64_t src =
              ptr_lds[e] + (uint64_t)(uint32_t)(lr.g - off_lds[e]) * (uint64_t)xrow_bytes;
          lr.src_lo = (uint32_t)src;
          lr.src_hi = (uint32_t)(src >> 32);
          lr.w_bits = __float_as_uint(load_weight(w, w_dtype, lr.g));
        } else {
          lr.src_lo = lr.src_hi = lr.w_bits = 0;
        }
        head += cnt;
        seen += cnt;
        add_rows<TX, V, U, R, AL>(lr, cnt, xrow_bytes, xoff, acc);
      }
      if (head > 0) {  // at most 63 rows carried to the window's front
        const int rest = have - head;
        const int carry = lane < rest ? win[wave][head + lane] : 0;
        if (lane < rest) win[wave][lane] = carry;
        have = rest;
      }
    }
    if (accumulate && seen == 0) continue;  // nothing routed here: out keeps its contents
#pragma unroll
    for (int u = 0; u < U; ++u)  // columns >= D: dropped by range check
      VO::template st<FMOE_OUT_CPOL>(ro, ooff[u], acc[u]);
  }
}

// ---- atomics ---------------------------------------------------------------------------------
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

template <typename TO, int V> struct AtomicVec;
template <int V> struct AtomicVec<float, V> {
  static __device__ __forceinline__ void add(float* p, const float* f) {
#pragma unroll
    for (int v = 0; v < V; ++v) unsafeAtomicAdd(p + v, f[v]);
  }
};
// 16-bit outputs: packed atomics on element pairs, so the vector path only (V even, rows and
// pairs 4-byte aligned); the host refuses atomic mode with a 16-bit output otherwise.
template <int V> struct AtomicVec<bf16_t, V> {
  static_assert(V % 2 == 0, "packed bf16 atomics need element pairs");
  static __device__ __forceinline__ void add(bf16_t* p, const float* f) {
#pragma unroll
    for (int v = 0; v < V; v += 2) {
      bf16x2_t x;
      x.x = (__bf16)f[v];
      x.y = (__bf16)f[v + 1];
      __builtin_amdgcn_global_atomic_fadd_v2bf16(reinterpret_cast<bf16x2_t*>(p + v), x);
    }
  }
};
template <int V> struct AtomicVec<f16_t, V> {
  static_assert(V % 2 == 0, "packed f16 atomics need element pairs");
  static __device__ __forceinline__ void add(f16_t* p, const float* f) {
#pragma unroll
    for (int v = 0; v < V; v += 2) {
      f16x2_t x;
      x.x = (_Float16)f[v];
      x.y = (_Float16)f[v + 1];
      __builtin_amdgcn_global_atomic_fadd_v2f16(reinterpret_cast<f16x2_t*>(p + v), x);
    }
  }
};

// Lane-interleaved row chunk: every access of the wave covers 64 * EPL consecutive columns (EPL =
// 1 for fp32 outputs, 2 for the packed 16-bit atomics), so the atomics of one instruction land on
// consecutive addresses -- two cache lines per instruction -- rather than on 16-byte lane strides
// spread over eight.  Device-scope float atomics are executed memory-side on MI355X (every L2
// atomic request is forwarded to the memory side), so the request count sets this kernel's speed.
// The chunk width (64 * V * U columns) is the one the host sized the grid with.
template <typename TX, typename TO, int V, int U, bool AL>
__device__ __forceinline__ void fwd_atomic_body(uint64_t src, float wf, TO* __restrict__ orow,
                                                uint32_t D, uint32_t chunk) {
  constexpr int EPL = sizeof(TO) == 4 ? 1 : 2;
  static_assert((V * U) % EPL == 0, "chunk must hold whole element pairs");
  constexpr int A = V * U / EPL;  // accesses per lane per chunk
  using VX = Vec<TX, EPL>;
  using raw_t = typename VX::raw_t;
  constexpr int CW = kWave * V * U;
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t col0 = chunk * CW + (uint32_t)lane * EPL;
  const rsrc_t rx = make_rsrc(src, D * (uint32_t)sizeof(TX));
  raw_t a[A];
#pragma unroll
  for (int i = 0; i < A; ++i)
    a[i] = load_x<TX, EPL, AL>(rx, (col0 + (uint32_t)i * kWave * EPL) * (uint32_t)sizeof(TX));
#pragma unroll
  for (int i = 0; i < A; ++i) {
    const uint32_t col = col0 + (uint32_t)i * kWave * EPL;
    float x[EPL];
    VX::cvt(a[i], x);
#pragma unroll
    for (int v = 0; v < EPL; ++v) x[v] = x[v] * wf;
    if (col < D) AtomicVec<TO, EPL>::add(orow + col, x);  // D is even for 16-bit outputs
  }
}

template <typename TX, typename TO, int V, int U>
__global__ __launch_bounds__(kGroup) void k_fwd_atomic(
    const int64_t* __restrict__ ptr_table, const int64_t* __restrict__ offsets, int64_t E,
    const void* __restrict__ idx, int idx_dtype, const void* __restrict__ w, int w_dtype,
    TO* __restrict__ out, int64_t out_stride, uint32_t D, uint32_t N, int64_t T, uint32_t chunks,
    int chunk_major) {
  constexpr int EPL = sizeof(TO) == 4 ? 1 : 2;
  const uint32_t unit = blockIdx.x * kWavesPerGroup + (uint32_t)uniform(threadIdx.x / kWave);
  uint32_t g, chunk;
  if (chunk_major) {  // every row's chunk 0, then every row's chunk 1, ...
    chunk = unit / N;
    if (chunk >= chunks) return;
    g = unit - chunk * N;
  } else {            // a row's chunks side by side
    g = unit / chunks;
    if (g >= N) return;
    chunk = unit - g * chunks;
  }
  const int64_t t = load_index(idx, idx_dtype, g);
  if (t < 0 || t >= T) return;  // out-of-range rows are dropped (the plan counts them)
  const int64_t e = expert_of_row(offsets, E, g);
  const uint64_t src =
      (uint64_t)ptr_table[e] + (uint64_t)((g - offsets[e]) * (int64_t)D) * sizeof(TX);
  const float wf = load_weight(w, w_dtype, g);
  TO* orow = out + t * out_stride;
  if (EPL > 1 && (src % (EPL * sizeof(TX))) != 0)
    fwd_atomic_body<TX, TO, V, U, false>(src, wf, orow, D, chunk);
  else
    fwd_atomic_body<TX, TO, V, U, true>(src, wf, orow, D, chunk);
}

// ---- atomic mode with few output rows: a workgroup's rows ordered by token first ----------------
// k_fwd_atomic sends every product to the memory side, whose atomic rate bounds it.  When the
// tokens are few, many of a workgroup's rows go to the same one: it takes a share of the rows and
// a slice of 64 columns, orders its rows by token in LDS (a counting sort; rows out of range are
// left out), and each of its waves walks a sixteenth of them, summing a token's run in registers
// and adding it to the output once.  The memory side then sees T + 15 adds per workgroup and
// column instead of its rows.  A lane holds one column, so that a wave's adds are consecutive (2
// and 4 columns per lane measured 67 and 198 us where 1 takes 58); 256 workgroups.  The sums start
// at -0, which a first term replaces exactly; the order of the additions varies, as everywhere in
// this mode.  us, k_fwd_atomic -> this kernel (one MI355X, three inputs in turn):
//   T=128, D=1024, N=65536   fp32 216 -> 58, bf16 211 -> 44      T=1000, D=1024, N=65536  212 -> 71
//   T=16, D=1024, N=65536    221 -> 52                           T=64, D=100, N=131072    83 -> 22
//   T=300, D=2048, N=131072  815 -> 224                          T=32, D=256, N=4096      9.6 -> 7.4
// Sums kept in LDS for all T tokens (ds_add_f32) took 341 us at the first of these: a wave's float
// add to LDS takes about 200 cycles.
constexpr int kFewThreads = kScanThreads;
constexpr int kFewWaves = kFewThreads / kWave;
constexpr int kFewGroups = 256;   // workgroups aimed at
constexpr int kFewRows = 8192;    // rows per workgroup at most: the sorted list's LDS
constexpr int kFewTokens = 1024;  // one per thread in the scan
constexpr int kFewBatch = 16;     // rows in flight per wave
static_assert(kFewRows <= (1 << 16) && kFewTokens <= (1 << 16), "list entries: token, row");
static_assert(kFewRows % kFewThreads == 0, "a thread keeps the tokens of its rows in registers");

template <typename TX>
__global__ __launch_bounds__(kFewThreads) void k_fwd_atomic_few(
    const int64_t* __restrict__ ptr_table, const int64_t* __restrict__ offsets, int64_t E,
    const void* __restrict__ idx, int idx_dtype, const void* __restrict__ w, int w_dtype,
    float* __restrict__ out, int64_t out_stride, uint32_t D, uint32_t N, uint32_t T,
    uint32_t slices, uint32_t rows_per_group) {
  using VX = Vec<TX, 1>;
  __shared__ uint32_t list[kFewRows];  // (token << 16 | row of the share), by token
  __shared__ int place[kFewTokens];    // rows per token, then the token's next place
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = uniform(tid / kWave);
  const uint32_t share = blockIdx.x / slices;  // of the rows; its slices are neighbours
  const uint32_t col = (blockIdx.x - share * slices) * kWave + (uint32_t)lane;
  const uint32_t beg = share * rows_per_group;  // < N: the host sizes the grid so
  const uint32_t n = min(rows_per_group, N - beg);
  place[tid] = 0;
  __syncthreads();
  // A row's index is read once and counted and placed from a register: the list has a place for
  // every row that was counted, whatever another stream does to the indices meanwhile.
  int tok[kFewRows / kFewThreads];  // -1: out of range, or no such row
#pragma unroll
  for (int j = 0; j < kFewRows / kFewThreads; ++j) {
    const uint32_t i = (uint32_t)(tid + j * kFewThreads);
    tok[j] = -1;
    if (i < n) {
      const int64_t t = load_index(idx, idx_dtype, beg + i);
      if (t >= 0 && t < (int64_t)T) tok[j] = (int)t;
    }
  }
#pragma unroll
  for (int j = 0; j < kFewRows / kFewThreads; ++j)
    if (tok[j] >= 0) atomicAdd(&place[tok[j]], 1);
  __syncthreads();
  int rows;
  const int first = block_exclusive_scan_1024(place[tid], &rows);
  place[tid] = first;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kFewRows / kFewThreads; ++j)
    if (tok[j] >= 0)
      list[atomicAdd(&place[tok[j]], 1)] =
          (uint32_t)tok[j] << 16 | (uint32_t)(tid + j * kFewThreads);
  __syncthreads();

  const uint32_t row_bytes = D * (uint32_t)sizeof(TX);
  const uint32_t off = col * (uint32_t)sizeof(TX);  // past the row: zeros from the range check
  const int per = (rows + kFewWaves - 1) / kFewWaves;
  const int p1 = min(rows, (wave + 1) * per);
  float acc = 0.f;
  int cur = -1;  // the token of acc; none yet
  auto flush = [&]() {
    if (cur >= 0 && col < D) unsafeAtomicAdd(out + (int64_t)cur * out_stride + col, acc);
  };
  for (int p = wave * per; p < p1; p += kWave) {
    const int cnt = min(kWave, p1 - p);
    LaneRecs lr;  // lr.g: the row's token
    lr.src_lo = lr.src_hi = lr.w_bits = 0;
    lr.g = -1;
    if (lane < cnt) {
      const uint32_t entry = list[p + lane];
      const int64_t g = beg + (entry & 0xffffu);
      const int64_t e = expert_of_row(offsets, E, g);
      const uint64_t src = (uint64_t)ptr_table[e] + (uint64_t)(g - offsets[e]) * row_bytes;
      lr.src_lo = (uint32_t)src;
      lr.src_hi = (uint32_t)(src >> 32);
      lr.w_bits = __float_as_uint(load_weight(w, w_dtype, g));
      lr.g = (int)(entry >> 16);
    }
    for (int i = 0; i < cnt; i += kFewBatch) {
      typename VX::raw_t a[kFewBatch];
#pragma unroll
      for (int r = 0; r < kFewBatch; ++r)
        a[r] = VX::template ld<FMOE_X_CPOL>(
            make_rsrc(lr.src(min(i + r, cnt - 1)), i + r < cnt ? row_bytes : 0u), off);
#pragma unroll
      for (int r = 0; r < kFewBatch; ++r) {
        if (i + r < cnt) {  // wave-uniform
          const int t = lr.row(i + r);
          if (t != cur) {  // wave-uniform
            flush();
            cur = t;
            acc = -0.f;
          }
          float x;
          VX::cvt(a[r], &x);
          acc = acc + x * lr.w(i + r);
        }
      }
    }
  }
  flush();
}

// ---- fp32 accumulator of a 16-bit output, and zero-fill of an overwritten output --------------
// Row-major passes over [T, D]: a thread per 8 consecutive columns of a row, with 16-byte accesses
// when the rows allow them (VEC: D % 8 == 0 and 16-byte aligned rows), element accesses otherwise.
// The accumulator is a contiguous, 16-byte aligned fp32 [T, D] workspace.
constexpr int kAccCols = 8;

template <typename TO, bool VEC>
__global__ __launch_bounds__(kGroup) void k_acc_init(float* __restrict__ acc,
                                                     const TO* __restrict__ out, int64_t out_stride,
                                                     uint32_t D, uint32_t T, int accumulate) {
  const uint32_t groups = (D + kAccCols - 1) / kAccCols;
  const int64_t total = (int64_t)T * groups;
  for (int64_t i = (int64_t)blockIdx.x * kGroup + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * kGroup) {
    const uint32_t t = (uint32_t)(i / groups);
    const uint32_t c = (uint32_t)(i - (int64_t)t * groups) * kAccCols;
    const TO* o = out + (int64_t)t * out_stride + c;
    float* a = acc + (int64_t)t * D + c;
    float f[kAccCols];
    if (!accumulate) {
#pragma unroll
      for (int k = 0; k < kAccCols; ++k) f[k] = 0.f;
    } else if constexpr (VEC) {
      Vec<TO, kAccCols>::cvt(*reinterpret_cast<const u32x4*>(o), f);
    } else {
#pragma unroll
      for (int k = 0; k < kAccCols; ++k) f[k] = c + k < D ? ld1(o + k) : 0.f;
    }
    if constexpr (VEC) {
      reinterpret_cast<u32x4*>(a)[0] = u32x4{__float_as_uint(f[0]), __float_as_uint(f[1]),
                                             __float_as_uint(f[2]), __float_as_uint(f[3])};
      reinterpret_cast<u32x4*>(a)[1] = u32x4{__float_as_uint(f[4]), __float_as_uint(f[5]),
                                             __float_as_uint(f[6]), __float_as_uint(f[7])};
    } else {
#pragma unroll
      for (int k = 0; k < kAccCols; ++k)
        if (c + k < D) a[k] = f[k];
    }
  }
}

template <typename TO, bool VEC>
__global__ __launch_bounds__(kGroup) void k_acc_store(const float* __restrict__ acc,
                                                      TO* __restrict__ out, int64_t out_stride,
                                                      uint32_t D, uint32_t T) {
  const uint32_t groups = (D + kAccCols - 1) / kAccCols;
  const int64_t total = (int64_t)T * groups;
  for (int64_t i = (int64_t)blockIdx.x * kGroup + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * kGroup) {
    const uint32_t t = (uint32_t)(i / groups);
    const uint32_t c = (uint32_t)(i - (int64_t)t * groups) * kAccCols;
    const float* a = acc + (int64_t)t * D + c;
    TO* o = out + (int64_t)t * out_stride + c;
    if constexpr (VEC) {
      const u32x4 lo = reinterpret_cast<const u32x4*>(a)[0];
      const u32x4 hi = reinterpret_cast<const u32x4*>(a)[1];
      const float f[kAccCols] = {__uint_as_float(lo.x), __uint_as_float(lo.y),
                                 __uint_as_float(lo.z), __uint_as_float(lo.w),
                                 __uint_as_float(hi.x), __uint_as_float(hi.y),
                                 __uint_as_float(hi.z), __uint_as_float(hi.w)};
      *reinterpret_cast<u32x4*>(o) = Vec<TO, kAccCols>::pack(f);
    } else {
#pragma unroll
      for (int k = 0; k < kAccCols; ++k)
        if (c + k < D) st1(o + k, a[k]);
    }
  }
}

// out[t, :] = 0 for every row (an atomic-mode call that overwrites out); 16-byte stores when
// the rows allow them (VEC, as in the accumulator passes).
template <typename TO, bool VEC>
__global__ __launch_bounds__(kGroup) void k_rows_zero(TO* __restrict__ out, int64_t out_stride,
                                                      uint32_t D, uint32_t T) {
  const uint32_t groups = (D + kAccCols - 1) / kAccCols;
  const int64_t total = (int64_t)T * groups;
  for (int64_t i = (int64_t)blockIdx.x * kGroup + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * kGroup) {
    const uint32_t t = (uint32_t)(i / groups);
    const uint32_t c = (uint32_t)(i - (int64_t)t * groups) * kAccCols;
    TO* o = out + (int64_t)t * out_stride + c;
    if constexpr (VEC) {
      constexpr int kWords = kAccCols * (int)sizeof(TO) / 16;  // 16-byte words per 8 columns
#pragma unroll
      for (int k = 0; k < kWords; ++k) reinterpret_cast<u32x4*>(o)[k] = u32x4{0u, 0u, 0u, 0u};
    } else {
#pragma unroll
      for (int k = 0; k < kAccCols; ++k)
        if (c + k < D) st1(o + k, 0.f);
    }
  }
}

static unsigned row_pass_blocks(int64_t T, int64_t D) {
  const int64_t threads = T * ((D + kAccCols - 1) / kAccCols);
  return (unsigned)std::min<int64_t>((threads + kGroup - 1) / kGroup, int64_t(1) << 16);
}

template <typename TO>
static int launch_zero(void* out, int64_t stride, int64_t D, int64_t T, hipStream_t s) {
  const bool vec = D % kAccCols == 0 && (uintptr_t)out % 16 == 0 &&
                   (stride * (int64_t)sizeof(TO)) % 16 == 0;
  if (vec)
    hipLaunchKernelGGL((k_rows_zero<TO, true>), dim3(row_pass_blocks(T, D)), dim3(kGroup), 0, s,
                       static_cast<TO*>(out), stride, (uint32_t)D, (uint32_t)T);
  else
    hipLaunchKernelGGL((k_rows_zero<TO, false>), dim3(row_pass_blocks(T, D)), dim3(kGroup), 0, s,
                       static_cast<TO*>(out), stride, (uint32_t)D, (uint32_t)T);
  return fmoe_host::check_launch("fmoe_combine_fwd(zero out)");
}

static int zero_out(void* out, int out_dtype, int64_t stride, int64_t D, int64_t T,
                    hipStream_t s) {
  if (out_dtype == FMOE_F32) return launch_zero<float>(out, stride, D, T, s);
  if (out_dtype == FMOE_BF16) return launch_zero<bf16_t>(out, stride, D, T, s);
  return launch_zero<f16_t>(out, stride, D, T, s);
}

template <typename TO>
static int launch_acc_pass(bool init, float* acc, void* out, int64_t stride, int64_t D, int64_t T,
                           int accumulate, hipStream_t s) {
  const bool vec = D % kAccCols == 0 && (uintptr_t)out % 16 == 0 &&
                   (stride * (int64_t)sizeof(TO)) % 16 == 0;
  const dim3 grid(row_pass_blocks(T, D));
  if (init) {
    if (vec)
      hipLaunchKernelGGL((k_acc_init<TO, true>), grid, dim3(kGroup), 0, s, acc,
                         static_cast<const TO*>(out), stride, (uint32_t)D, (uint32_t)T, accumulate);
    else
      hipLaunchKernelGGL((k_acc_init<TO, false>), grid, dim3(kGroup), 0, s, acc,
                         static_cast<const TO*>(out), stride, (uint32_t)D, (uint32_t)T, accumulate);
  } else {
    if (vec)
      hipLaunchKernelGGL((k_acc_store<TO, true>), grid, dim3(kGroup), 0, s, acc,
                         static_cast<TO*>(out), stride, (uint32_t)D, (uint32_t)T);
    else
      hipLaunchKernelGGL((k_acc_store<TO, false>), grid, dim3(kGroup), 0, s, acc,
                         static_cast<TO*>(out), stride, (uint32_t)D, (uint32_t)T);
  }
  return fmoe_host::check_launch("fmoe_combine_fwd(fp32 accumulator)");
}

// ---- host dispatch ---------------------------------------------------------------------------
// Vectors per lane per row: several 16-byte loads in flight per row, and preferably a chunk
// width that divides D (no tail predication), while small D still spreads over many waves.
static int pick_u(int64_t D, int V) {
  const int forced = (int)fmoe_host::opt(fmoe_host::kOptFwdDetU);
  if (forced == 1 || forced == 2 || forced == 4) return forced;
  for (int u = 4; u >= 1; u >>= 1) {
    const int64_t cw = (int64_t)kWave * V * u;
    if (D % cw == 0 && D / cw >= (u == 1 ? 1 : 2)) return u;
  }
  if (D >= (int64_t)kWave * V * 4 * 2) return 4;
  if (D >= (int64_t)kWave * V * 2) return 2;
  return 1;
}

static int grid_for(int64_t units, const char* who, unsigned* blocks) {
  const int64_t b = (units + kWavesPerGroup - 1) / kWavesPerGroup;
  if (units >= (int64_t(1) << 32) - kWavesPerGroup || b >= (int64_t(1) << 31)) {
    fmoe_host::set_error("%s: grid too large (%lld wave units)", who, (long long)units);
    return FMOE_ERANGE;
  }
  *blocks = (unsigned)b;
  return FMOE_OK;
}

struct FwdArgs {
  int mode;
  bool step;  // FMOE_MODE_DET_STEP
  const int32_t* status;
  const int32_t* row_ptr;
  const Rec* rec;
  const void* idx;
  int idx_dtype;
  const void* w;
  int w_dtype;
  const int64_t* ptr_table;
  const int64_t* offsets;
  int64_t E, N, T, D;
  void* out;
  int64_t out_stride;
  int accumulate;
  unsigned lds;  // dynamic LDS of the deterministic kernel (DetTile)
  hipStream_t s;
};

// Whether the deterministic forward stores its output non-temporally.  Stored with the temporal
// policy (FMOE_OUT_CPOL), the output stays dirty in the 256 MB Infinity Cache: the forward itself is
// shorter if the output's lines are still there from the call before (a loop that writes the same
// buffer), but they are written back during the kernels that follow, which loses more once the output
// is a large part of that cache.  Time non-temporal / temporal, bf16 but for the last row (one MI355X,
// three sets of inputs; the forward alone into one buffer | into three in turn | with its backward):
//   T, D (output)              top-1                top-3                top-8
//   12288, 4096 (96 MiB)       1.11 | 1.03 | 0.99   1.07 | 0.97 | 0.94   1.01 | 0.94 | 0.95
//   16384, 4096 (128 MiB)      1.11 | 0.98 | 0.92   1.05 | 0.97 | 0.95   1.01 | 0.96 | 0.96
//   4096, 16384 (128 MiB)      1.13 | 0.97 | 0.97   1.06 | 0.97 | 0.94   1.02 | 0.99 | 0.96
//   16384, 7168 (224 MiB)      1.17 | 1.00 | 0.92   1.08 | 0.99 | 0.93   1.01 | 1.00 | 0.94
//   16384, 12288 (384 MiB)     1.00 | 1.00 | 0.99   1.00 | 1.01 | 0.95
//   fp32 8192, 8192 (256 MiB)  1.15 | 0.98 | 0.95   1.07 | 0.99 | 0.91   1.06 | 1.01 | 0.93
// So a forward whose backward follows streams from 96 MiB, and one alone only from 7 rows per token,
// where it gains as much in a program that goes on to other buffers as it loses in one that does not.
// Steps below that line (2048, 16384, top-8, 64 MiB: 313.7 -> 297.5 us) stay temporal with the
// forwards.  An accumulating call has just read its output and the caller has just written it, so its
// lines are in the cache: fp32, 256 MiB, zero-fill + call 291.6 us temporal, 316.9 us non-temporal;
// it stays temporal.
static int streams_out(const FwdArgs& a, int64_t elem_bytes) {
  return !a.accumulate && a.T * a.D * elem_bytes >= FMOE_STREAM_OUT_BYTES &&
         (a.step || a.N >= 7 * a.T);
}

template <typename TX, typename TO, int V, int U, int RB>
static int launch_fwd_k(const FwdArgs& a, int64_t chunks) {
  unsigned blocks;
  if (a.mode == FMOE_MODE_DET) {
    if (int rc = grid_for(a.T * chunks, "fmoe_combine_fwd(det)", &blocks)) return rc;
    const int persist = (int)fmoe_host::opt(fmoe_host::kOptFwdGrid);  // 0 = one wave per unit
    if (persist > 0 && (unsigned)persist < blocks) blocks = (unsigned)persist;
    hipLaunchKernelGGL((k_fwd_det<TX, TO, V, U, RB>), dim3(blocks), dim3(kGroup), a.lds, a.s,
                       a.status, a.row_ptr, a.rec, static_cast<TO*>(a.out), a.out_stride,
                       (uint32_t)a.D, (uint32_t)a.T, (uint32_t)chunks, a.accumulate,
                       streams_out(a, sizeof(TO)));
    return fmoe_host::check_launch("fmoe_combine_fwd(det)");
  }
  if constexpr (V == 1 && sizeof(TO) == 2) {
    fmoe_host::set_error(
        "fmoe_combine_fwd(atomic_packed): a 16-bit output needs D %% %d == 0 and %d-byte aligned "
        "output rows (packed atomics on element pairs); use FMOE_MODE_ATOMIC or FMOE_MODE_DET",
        vec16<TX>(), vec16<TX>() * 2);
    return FMOE_EINVAL;
  } else {
    if (int rc = grid_for(a.N * chunks, "fmoe_combine_fwd(atomic)", &blocks)) return rc;
    // Column-chunk-major order keeps each pass over the rows on one column slice of the target.
    // Measured (rocprof, one MI355X, bf16 experts, fp32 accumulator): with a 2 GiB target
    // (T = 32768, D = 16384, top-2) the atomic kernel takes 3332 against 3381 us; with 256 MiB
    // targets (T = 4096, D = 16384, top-8; T = 8192, D = 4096, top-6) it is 1-1.5 % slower, so it
    // is the default from 1 GiB of target.
    const int order = (int)fmoe_host::opt(fmoe_host::kOptAtomicOrder);
    const bool big = a.T * a.D * (int64_t)sizeof(TO) >= (int64_t(1) << 30);
    const int chunk_major = (order == 2 || (order == 0 && big)) ? 1 : 0;
    hipLaunchKernelGGL((k_fwd_atomic<TX, TO, V, U>), dim3(blocks), dim3(kGroup), 0, a.s,
                       a.ptr_table, a.offsets, a.E, a.idx, a.idx_dtype, a.w, a.w_dtype,
                       static_cast<TO*>(a.out), a.out_stride, (uint32_t)a.D, (uint32_t)a.N, a.T,
                       (uint32_t)chunks, chunk_major);
    return fmoe_host::check_launch("fmoe_combine_fwd(atomic)");
  }
}

template <typename TX, typename TO, int V, int U, int RB>
static int launch_fwd_u(const FwdArgs& a) {
  const int64_t CW = (int64_t)kWave * V * U;
  const int64_t chunks = (a.D + CW - 1) / CW;
  return launch_fwd_k<TX, TO, V, U, RB>(a, chunks);
}

// Tile of the deterministic forward: U vectors per lane per row, R rows per batch, and `lds` bytes
// of unused dynamic LDS, which bound the workgroups resident on a CU.
struct DetTile {
  int U, R;
  unsigned lds;
};
// The most LDS that still lets `groups` workgroups share a CU's 160 KB, which is handed out in
// pieces of 1280 bytes.
constexpr unsigned lds_for_groups(int groups) { return (160u << 10) / 1280 / groups * 1280; }

// The choice by the rows per token r = N / T and the bytes of the rows.
//
// Short segments.  A batch issues its R x U loads whether or not its rows exist (the spare slots
// read an empty range: no traffic, but an issue slot each), so r <= 1.5 takes R = 2 (U = 4, with a
// partly empty last chunk if D needs it, when D holds one chunk of 4 vectors per lane) and r < 2.5
// takes R = 4.  bf16, T=16384, D=7168, us against the choice by D alone: k=1 129 -> 75, k=2 146 ->
// 109.
//
// Longer segments are bound by how HBM serves thousands of row pieces read side by side, and lose
// rate when more of them are in flight than its latency needs (64 to 96 KB of loads per CU).  Rows
// that the 256 MB Infinity Cache cannot hold therefore take U = 2, R = 4 with 4 resident workgroups
// per CU for r < 3.5, 3 beyond, and 2 for r >= 7 from 768 MB; smaller ones, which finish in a few
// rounds, take U = 4, R = 2 with every slot in use.  bf16 (three sets of buffers in turn, us, the
// previous choice -> this one; the same tile without the bound in brackets):
//   T=4096, D=16384, k=8   208.2 -> 198.5 (212.8)     T=8192, D=16384, k=6   325.0 -> 308.8 (346.2)
//   T=16384, D=7168, k=8   374.4 -> 348.8 (379.2)     T=8192, D=16384, k=5   272.0 -> 260.9 (286.3)
//   T=16384, D=4096, k=8   211.2 -> 199.9 (214.8)     T=16384, D=16384, k=4  461.5 -> 429.1 (466.5)
//   T=8192, D=4096, k=6     76.5 ->  75.6 ( 76.9)     T=16384, D=7168, k=3   157.4 -> 149.1 (157.5)
//   T=4096, D=8192, k=8     99.6 ->  96.7 ( 99.6)     T=8192, D=3072, k=8     75.7 ->  73.7 ( 75.7)
//   T=1024, D=7168, k=8     25.2 ->  23.4             T=512, D=7168, k=8      13.3 ->  11.9
//   fp32: T=4096, D=16384, k=8  427.4 -> 404.0 (433.4); k=4  227.7 -> 215.7 (224.9)
// With 2 workgroups T=8192, D=4096, k=6 takes 81.7 us and T=4096, D=8192, k=8 98.1; r < 2.5 loses
// under every bound (T=8192, D=4096, k=2: 31.9, 36.7 with 3 workgroups).
//
// Few wave units.  A wider tile makes fewer of them, and below 1280 (U = 4; 1024 for U = 2), five or
// four to a CU, the waves missing cost more than the tile gains, at every size of the rows: those
// calls keep the tile by D and r (narrow_det_tile), where U = 4 gives way to U = 2 below 512 wave
// units.  The kernel alone, bf16, us, the tile above / the tile by D and r, wave units of the former:
//   T=256, D=2048, k=8:   256,  7.0 /  4.6     T=512, D=2048, k=8:    512,  7.4 /  5.8
//   T=256, D=1536, k=8:   512,  5.0 /  4.4     T=512, D=4096, k=4:   1024,  6.0 /  5.4
//   T=1024, D=4096, k=8: 2048, 13.7 / 14.1     T=1024, D=3072, k=4:  2048,  7.4 /  7.6
//   N=131072: T=64, D=1024: 64, 506 / 362      T=16, D=4096: 64, 1961 / 3169 with U = 4
static DetTile narrow_det_tile(int64_t N, int64_t T, int64_t D, int V) {
  DetTile c{pick_u(D, V), 0, 0};
  c.R = c.U >= 4 ? 4 : 8;
  if (2 * N < 7 * T) {
    if (c.U >= 2) c.R = 4;
  } else if (c.U == 4) {
    const int64_t CW = (int64_t)kWave * V * 4;
    if (T * ((D + CW - 1) / CW) < 512) c = {2, 4, 0};
  } else if (N >= 7 * T && c.U == 2) {
    c = {1, 8, 0};
  }
  return c;
}

static DetTile pick_det_tile(int64_t N, int64_t T, int64_t D, int64_t x_bytes, int V) {
  DetTile c{pick_u(D, V), 0, 0};
  c.R = c.U >= 4 ? 4 : 8;
  if (fmoe_host::opt(fmoe_host::kOptFwdDetU) != 0 || N == 0) return c;  // U forced: keep R by U
  const int64_t bytes = N * D * x_bytes;
  if (2 * N <= 3 * T && D >= (int64_t)kWave * V * 4) return {4, 2, 0};  // r <= 1.5
  if (2 * N < 5 * T) return narrow_det_tile(N, T, D, V);                // r < 2.5
  if (D < (int64_t)kWave * V * 2) return c;  // less than a chunk of 2 vectors per lane
  if (bytes >= (int64_t(256) << 20)) {
    const bool two = N >= 7 * T && bytes >= (int64_t(768) << 20);
    c = {2, 4, lds_for_groups(2 * N < 7 * T ? 4 : (two ? 2 : 3))};
  } else if (2 * N < 7 * T) {  // r < 3.5
    return narrow_det_tile(N, T, D, V);
  } else if (D >= (int64_t)kWave * V * 4) {
    c = {4, 2, 0};
  } else {
    c = {2, 4, 0};
  }
  const int64_t CW = (int64_t)kWave * V * c.U;
  return T * ((D + CW - 1) / CW) < (c.U == 4 ? 1280 : 1024) ? narrow_det_tile(N, T, D, V) : c;
}

// Tile shapes (U vectors per lane per row, R rows per batch).  The "fwd_tile" option <U><R> (e.g.
// 44) overrides the choice for tuning.
template <typename TX, typename TO, int V>
static int launch_fwd_v(FwdArgs a) {
  if constexpr (V == 1) {
    return launch_fwd_u<TX, TO, 1, 4, 4>(a);
  } else {
    const int tile = (int)fmoe_host::opt(a.mode == FMOE_MODE_DET ? fmoe_host::kOptFwdTile
                                                                 : fmoe_host::kOptFwdAtomicTile);
    int U = tile / 10, R = tile % 10;
    if (!((U == 4 && (R == 4 || R == 2)) || (U == 2 && (R == 8 || R == 4)) ||
          (U == 1 && R == 8))) {
      if (a.mode == FMOE_MODE_DET) {
        const DetTile c = pick_det_tile(a.N, a.T, a.D, sizeof(TX), V);
        U = c.U;
        R = c.R;
        a.lds = c.lds;
      } else {
        U = pick_u(a.D, V);
        R = U >= 4 ? 4 : 8;
      }
    }
    if (U == 4 && R == 2) return launch_fwd_u<TX, TO, V, 4, 2>(a);
    if (U == 4) return launch_fwd_u<TX, TO, V, 4, 4>(a);
    if (U == 2 && R == 4) return launch_fwd_u<TX, TO, V, 2, 4>(a);
    if (U == 2) return launch_fwd_u<TX, TO, V, 2, 8>(a);
    return launch_fwd_u<TX, TO, V, 1, 8>(a);
  }
}

// The few-tokens atomic kernel: its geometry, or 0 groups where it is not taken.  It takes an fp32
// target (a 16-bit output's accumulator among them) of at most kFewTokens rows.  Its shares hold 4
// rows per token or more, so that the ordering saves atomics; where that leaves few workgroups, or
// little work, the ordering costs more than the atomics of k_fwd_atomic, which spreads the same rows
// over the whole device.  So the rule asks for 64 workgroups and for N * D >= 2^22, 2^20 from 96
// workgroups, or 2^19 from 256 rows per token, whose atomics queue at an address.  us, k_fwd_atomic /
// this kernel, fp32, whole calls (one MI355X, three inputs in turn):
//   workgroups: T=1024, N=6144, D=64: 1, 7.9 / 65     T=1024, N=8192, D=512: 16, 21.0 / 51.9
//     T=1024, N=16384, D=512: 32, 34.7 / 53.5         T=512, N=6144, D=1024: 48, 28.3 / 31.3
//     T=512, N=8192, D=1024: 64, 35.0 / 31.9          T=256, N=1536, D=4096: 64, 28.9 / 26.0
//     T=512, N=6144, D=2048: 96, 48.5 / 34.1          T=1024, N=16384, D=2048: 128, 113 / 60.1
//   work, 64 workgroups: 2^20 (T=64, N=1024, D=1024) 10.0 / 11.2; 2^21 (T=128, N=1024, D=2048)
//     13.5 / 13.7; 2^22 (T=256, N=2048, D=2048) 21.6 / 20.4
//   work, 128 and more: 2^19 (T=16, N=256, D=2048) 9.6 / 10.2; 2^20 (T=16, N=512, D=2048) 12.1 / 10.5
//   256 rows per token: T=1, N=256, D=1024 14.1 / 15.1, D=2048 16.7 / 12.2
// Option "fwd_atomic_few": 1 = never, 2 = whenever the tokens fit.  A forced tile or grid order of
// k_fwd_atomic turns it off.
struct FewGeom {
  int64_t slices, rows_per_group, groups;
};
static FewGeom few_geom(int64_t N, int64_t T, int64_t D) {
  FewGeom g{};
  const int64_t choice = fmoe_host::opt(fmoe_host::kOptAtomicFew);
  if (N < 1 || T < 1 || T > kFewTokens || D < 1 || choice == 1 ||
      fmoe_host::opt(fmoe_host::kOptFwdAtomicTile) != 0 ||
      fmoe_host::opt(fmoe_host::kOptAtomicOrder) != 0)
    return g;
  g.slices = (D + kWave - 1) / kWave;
  int64_t shares = std::max<int64_t>(1, kFewGroups / g.slices);
  shares = std::min<int64_t>(shares, N / (4 * T));
  shares = std::max<int64_t>(shares, (N + kFewRows - 1) / kFewRows);
  g.rows_per_group = (N + shares - 1) / shares;
  shares = (N + g.rows_per_group - 1) / g.rows_per_group;  // none of them empty
  const int64_t groups = shares * g.slices;
  const int work_bits = N >= 256 * T ? 19 : (groups >= 96 ? 20 : 22);
  if (choice == 2 || (N >= 4 * T && groups >= 64 && N * D >= (int64_t(1) << work_bits)))
    g.groups = groups;
  return g;
}

template <typename TX>
static int launch_few(const FwdArgs& a, const FewGeom& g) {
  if (g.groups >= (int64_t(1) << 31)) {
    fmoe_host::set_error("fmoe_combine_fwd(atomic): grid too large (%lld workgroups)",
                         (long long)g.groups);
    return FMOE_ERANGE;
  }
  hipLaunchKernelGGL((k_fwd_atomic_few<TX>), dim3((unsigned)g.groups), dim3(kFewThreads), 0, a.s,
                     a.ptr_table, a.offsets, a.E, a.idx, a.idx_dtype, a.w, a.w_dtype,
                     static_cast<float*>(a.out), a.out_stride, (uint32_t)a.D, (uint32_t)a.N,
                     (uint32_t)a.T, (uint32_t)g.slices, (uint32_t)g.rows_per_group);
  return fmoe_host::check_launch("fmoe_combine_fwd(atomic, few tokens)");
}

template <typename TX, typename TO>
static int launch_fwd_t(const FwdArgs& a) {
  if constexpr (sizeof(TO) == 4) {
    if (a.mode != FMOE_MODE_DET) {
      const FewGeom g = few_geom(a.N, a.T, a.D);
      if (g.groups > 0) return launch_few<TX>(a, g);
    }
  }
  constexpr int V = vec16<TX>();
  const int ob = (int)sizeof(TO) == 4 ? 4 : 2;
  const int64_t vb = (int64_t)V * ob;  // bytes of one output vector
  const bool vec_ok = (a.D % V == 0) && ((uintptr_t)a.out % vb == 0) &&
                      ((a.out_stride * ob) % vb == 0) && fmoe_host::opt(fmoe_host::kOptForceScalar) == 0;
  if (vec_ok) return launch_fwd_v<TX, TO, V>(a);
  return launch_fwd_v<TX, TO, 1>(a);
}

template <typename TX>
static int launch_fwd_x(const FwdArgs& a, int out_dtype) {
  switch (out_dtype) {
    case FMOE_F32: return launch_fwd_t<TX, float>(a);
    case FMOE_BF16: return launch_fwd_t<TX, bf16_t>(a);
    case FMOE_F16: return launch_fwd_t<TX, f16_t>(a);
  }
  fmoe_host::set_error("fmoe_combine_fwd: bad out dtype %d", out_dtype);
  return FMOE_EINVAL;
}


// The dispatch permutation's backward: k_fwd_det's tiles over the packed-row gradients.
struct SlotsBwdArgs {
  const int32_t* slot_pos;
  int64_t T, k, D;
  const void* rows;
  void* out;
  const void* gates;
  void* grad_gates;
  hipStream_t s;
  unsigned lds;  // DetTile
};

// grad_x is streamed from a smaller size than the forward's output (streams_out): a backward is
// always followed by more passes over as much data, which pay for the lines left in the cache.
// Permutation forward + backward, three sets of buffers in turn, bf16, temporal / non-temporal:
// T=8192, D=4096, top-6 and T=4096, D=8192, top-6 (64 MiB) 180.9 / 165.9 and 182.0 / 164.8 us;
// 28 and 32 MiB of grad_x make no difference.  Where the program frees each result at once, so that
// the next call's buffers are the same lines, forward + backward hardly changes up to 128 MiB and
// gains beyond; time non-temporal / temporal where the GPU bounds the call:
//   8192, 4096 (64 MiB)    top-6 0.99, top-8 1.00
//   12288, 4096 (96 MiB)   top-4 1.00, top-6 1.00, top-8 1.01
//   16384, 4096 (128 MiB)  top-2 1.04, top-4 1.01, top-6 1.02, top-8 1.01
//   16384, 7168 (224 MiB)  top-1 0.95, top-2 0.96, top-4 0.96, top-6 0.98, top-8 0.98
//   16384, 16384 (512 MiB) top-1 0.95, top-2 0.95, top-4 0.95
// (the backward alone, over and over, loses 2 to 5 % there, and 3 to 19 % at 224 MiB).
constexpr int64_t kSlotsStreamBytes = int64_t(48) << 20;

template <typename TX, int V, int U, int RB, bool GATES, typename TG>
static int launch_slots_bwd_k(const SlotsBwdArgs& a) {
  const int64_t CW = (int64_t)kWave * V * U;
  const int64_t chunks = (a.D + CW - 1) / CW;
  unsigned blocks;
  if (int rc = grid_for(a.T * chunks, "fmoe_permute_backward", &blocks)) return rc;
  hipLaunchKernelGGL((k_slots_bwd<TX, V, U, RB, GATES, TG>), dim3(blocks), dim3(kGroup), a.lds, a.s,
                     a.slot_pos, (uint32_t)a.k, (uint32_t)(a.T * a.k),
                     static_cast<const TX*>(a.rows), (uint32_t)a.D, (uint32_t)a.T,
                     (uint32_t)chunks, static_cast<TX*>(a.out),
                     a.T * a.D * (int64_t)sizeof(TX) >= kSlotsStreamBytes,
                     static_cast<const TG*>(a.gates), static_cast<TG*>(a.grad_gates));
  return fmoe_host::check_launch("fmoe_permute_backward");
}

template <typename TX, int V, int U, int RB>
static int launch_slots_bwd_g(const SlotsBwdArgs& a, int gate_dtype) {
  if (!a.grad_gates) return launch_slots_bwd_k<TX, V, U, RB, false, uint32_t>(a);
  if (fmoe_host::dtype_bytes(gate_dtype) == 4)
    return launch_slots_bwd_k<TX, V, U, RB, true, uint32_t>(a);
  return launch_slots_bwd_k<TX, V, U, RB, true, uint16_t>(a);
}

// 16-byte vectors when every row is 16-byte aligned, else one element per lane.
template <typename TX>
static int launch_slots_bwd(SlotsBwdArgs a, int gate_dtype) {
  constexpr int V = vec16<TX>();
  const bool vec_ok = a.D % V == 0 && (uintptr_t)a.rows % 16 == 0 && (uintptr_t)a.out % 16 == 0 &&
                      fmoe_host::opt(fmoe_host::kOptForceScalar) == 0;
  if (!vec_ok) return launch_slots_bwd_g<TX, 1, 4, 4>(a, gate_dtype);
  const DetTile c = pick_det_tile(a.T * a.k, a.T, a.D, sizeof(TX), V);
  a.lds = c.lds;
  if (c.U == 4 && c.R == 2) return launch_slots_bwd_g<TX, V, 4, 2>(a, gate_dtype);
  if (c.U == 4) return launch_slots_bwd_g<TX, V, 4, 4>(a, gate_dtype);
  if (c.U == 2 && c.R == 4) return launch_slots_bwd_g<TX, V, 2, 4>(a, gate_dtype);
  if (c.U == 2) return launch_slots_bwd_g<TX, V, 2, 8>(a, gate_dtype);
  return launch_slots_bwd_g<TX, V, 1, 8>(a, gate_dtype);
}

// The small path: a grid of at most kSmallGroups workgroups strides over the (token, chunk) units,
// so that the ids are staged at most that many times.
constexpr unsigned kSmallGroups = 1024;

struct SmallFwdArgs {
  HostTable meta;
  const void* idx;
  int idx_dtype;
  const void* w;
  int w_dtype;
  int64_t N, T, D;
  void* out;
  int64_t out_stride;
  int accumulate;
  int32_t* status;
  bool aligned;
  hipStream_t s;
};

template <typename TX, typename TO, int V, int U, bool AL>
static int launch_small_k(const SmallFwdArgs& a) {
  const int64_t CW = (int64_t)kWave * V * U;
  const int64_t chunks = (a.D + CW - 1) / CW;
  unsigned blocks;
  if (int rc = grid_for(a.T * chunks, "fmoe_combine_fwd_small", &blocks)) return rc;
  blocks = std::min(blocks, kSmallGroups);
  hipLaunchKernelGGL((k_fwd_small<TX, TO, V, U, AL>), dim3(blocks), dim3(kGroup), 0, a.s, a.meta,
                     a.idx, a.idx_dtype, a.w, a.w_dtype, (uint32_t)a.N, (uint32_t)a.T,
                     (uint32_t)a.D, (uint32_t)chunks, static_cast<TO*>(a.out), a.out_stride,
                     a.accumulate, a.status);
  return fmoe_host::check_launch("fmoe_combine_fwd_small");
}

// 16-byte vectors when the output layout allows them (as launch_fwd_t), U by D (pick_u); rows
// that are not 16-byte aligned take element loads one vector per lane.
template <typename TX, typename TO>
static int launch_small_t(const SmallFwdArgs& a) {
  constexpr int V = vec16<TX>();
  const int ob = (int)sizeof(TO) == 4 ? 4 : 2;
  const int64_t vb = (int64_t)V * ob;
  const bool vec_ok = (a.D % V == 0) && ((uintptr_t)a.out % vb == 0) &&
                      ((a.out_stride * ob) % vb == 0) &&
                      fmoe_host::opt(fmoe_host::kOptForceScalar) == 0;
  if (!vec_ok) return launch_small_k<TX, TO, 1, 4, true>(a);
  if (!a.aligned) return launch_small_k<TX, TO, V, 1, false>(a);
  const int U = pick_u(a.D, V);
  if (U == 4) return launch_small_k<TX, TO, V, 4, true>(a);
  if (U == 2) return launch_small_k<TX, TO, V, 2, true>(a);
  return launch_small_k<TX, TO, V, 1, true>(a);
}

template <typename TX>
static int launch_small_x(const SmallFwdArgs& a, int out_dtype) {
  switch (out_dtype) {
    case FMOE_F32: return launch_small_t<TX, float>(a);
    case FMOE_BF16: return launch_small_t<TX, bf16_t>(a);
    case FMOE_F16: return launch_small_t<TX, f16_t>(a);
  }
  fmoe_host::set_error("fmoe_combine_fwd_small: bad out dtype %d", out_dtype);
  return FMOE_EINVAL;
}

}  // namespace fmoe

extern "C" int64_t fmoe_combine_fwd_workspace_bytes(int mode, int64_t num_tokens, int64_t hidden,
                                                    int out_dtype) {
  if (num_tokens < 1 || hidden < 1) return -1;
  if (mode == FMOE_MODE_ATOMIC && (out_dtype == FMOE_BF16 || out_dtype == FMOE_F16))
    return fmoe_host::round_up(num_tokens * hidden * 4, 256);
  return 0;
}

extern "C" int fmoe_combine_fwd(int mode, const void* d_plan, const void* d_indices, int idx_dtype,
                                const void* d_weights, int w_dtype, const int64_t* d_ptr_table,
                                const int64_t* d_offsets, int64_t num_experts, int64_t num_rows,
                                int64_t num_tokens, int64_t hidden, int x_dtype, void* d_out,
                                int out_dtype, int64_t out_row_stride, int accumulate,
                                void* d_workspace, int64_t workspace_bytes, void* stream) {
  using namespace fmoe;
  fmoe_host::clear_error();
  const bool step = mode == FMOE_MODE_DET_STEP;
  if (step) mode = FMOE_MODE_DET;
  FMOE_REQUIRE(mode == FMOE_MODE_DET || mode == FMOE_MODE_ATOMIC || mode == FMOE_MODE_ATOMIC_PACKED,
               "fmoe_combine_fwd: bad mode %d", mode);
  FMOE_REQUIRE(num_rows >= 0 && num_tokens >= 1 && hidden >= 1,
               "fmoe_combine_fwd: bad sizes N=%lld T=%lld D=%lld", (long long)num_rows,
               (long long)num_tokens, (long long)hidden);
  if (num_rows >= (int64_t(1) << 31) || num_tokens >= (int64_t(1) << 30)) {
    fmoe_host::set_error("fmoe_combine_fwd: N/T exceed the 32-bit row counters");
    return FMOE_ERANGE;
  }
  FMOE_REQUIRE(fmoe_host::is_float_dtype(x_dtype), "fmoe_combine_fwd: bad x dtype %d", x_dtype);
  FMOE_REQUIRE(fmoe_host::is_float_dtype(out_dtype), "fmoe_combine_fwd: bad out dtype %d",
               out_dtype);
  FMOE_REQUIRE(d_out != nullptr, "fmoe_combine_fwd: null out");
  FMOE_REQUIRE(out_row_stride >= hidden, "fmoe_combine_fwd: out row stride %lld < D %lld",
               (long long)out_row_stride, (long long)hidden);
  if (hidden * 4 >= (int64_t(1) << 31)) {
    fmoe_host::set_error("fmoe_combine_fwd: D=%lld exceeds the 2 GiB row limit", (long long)hidden);
    return FMOE_ERANGE;
  }
  FwdArgs a{};
  a.mode = mode;
  a.step = step;
  a.N = num_rows;
  a.T = num_tokens;
  a.D = hidden;
  a.E = num_experts;
  a.out = d_out;
  a.out_stride = out_row_stride;
  a.accumulate = accumulate ? 1 : 0;
  a.s = static_cast<hipStream_t>(stream);
  if (mode == FMOE_MODE_DET) {
    FMOE_REQUIRE(d_plan != nullptr, "fmoe_combine_fwd(det): null plan");
    FMOE_REQUIRE(((uintptr_t)d_plan & 255) == 0, "fmoe_combine_fwd(det): plan not 256B-aligned");
    const char* ws = static_cast<const char*>(d_plan);
    a.status = reinterpret_cast<const int32_t*>(ws + fmoe_plan_status_offset());
    a.row_ptr = reinterpret_cast<const int32_t*>(ws + fmoe_plan_row_ptr_offset(a.N, a.T));
    a.rec = reinterpret_cast<const Rec*>(ws + fmoe_plan_records_offset(a.N, a.T));
    switch (x_dtype) {
      case FMOE_F32: return launch_fwd_x<float>(a, out_dtype);
      case FMOE_BF16: return launch_fwd_x<bf16_t>(a, out_dtype);
      case FMOE_F16: return launch_fwd_x<f16_t>(a, out_dtype);
    }
    fmoe_host::set_error("fmoe_combine_fwd: bad x dtype %d", x_dtype);
    return FMOE_EINVAL;
  }
  // atomic modes: the fp32 accumulator of a 16-bit output first (its size is checked before any
  // launch)
  const bool acc16 = mode == FMOE_MODE_ATOMIC && out_dtype != FMOE_F32;
  const int64_t need = fmoe_combine_fwd_workspace_bytes(mode, num_tokens, hidden, out_dtype);
  if (acc16)
    FMOE_REQUIRE(d_workspace && workspace_bytes >= need && ((uintptr_t)d_workspace & 15) == 0,
                 "fmoe_combine_fwd(atomic): a 16-bit output needs a 16-byte aligned fp32 "
                 "workspace of %lld bytes (fmoe_combine_fwd_workspace_bytes), got %lld",
                 (long long)need, (long long)workspace_bytes);
  if (num_rows == 0)  // nothing to add: an overwrite still clears out
    return accumulate ? FMOE_OK : zero_out(d_out, out_dtype, out_row_stride, hidden, num_tokens, a.s);
  FMOE_REQUIRE(d_indices && d_weights && d_ptr_table && d_offsets,
               "fmoe_combine_fwd(atomic): null index/weight/metadata pointer");
  FMOE_REQUIRE(fmoe_host::is_index_dtype(idx_dtype), "fmoe_combine_fwd: bad index dtype %d",
               idx_dtype);
  FMOE_REQUIRE(fmoe_host::is_float_dtype(w_dtype), "fmoe_combine_fwd: bad weight dtype %d",
               w_dtype);
  FMOE_REQUIRE(num_experts >= 1, "fmoe_combine_fwd: num_experts must be >= 1");
  a.idx = d_indices;
  a.idx_dtype = idx_dtype;
  a.w = d_weights;
  a.w_dtype = w_dtype;
  a.ptr_table = d_ptr_table;
  a.offsets = d_offsets;
  int target_dtype = out_dtype;
  float* acc = static_cast<float*>(d_workspace);
  if (acc16) {
    const int rc = out_dtype == FMOE_BF16
                       ? launch_acc_pass<bf16_t>(true, acc, d_out, out_row_stride, hidden,
                                                 num_tokens, accumulate, a.s)
                       : launch_acc_pass<f16_t>(true, acc, d_out, out_row_stride, hidden,
                                                num_tokens, accumulate, a.s);
    if (rc) return rc;
    a.out = acc;
    a.out_stride = hidden;
    target_dtype = FMOE_F32;
  } else if (!accumulate) {
    if (int rc = zero_out(d_out, out_dtype, out_row_stride, hidden, num_tokens, a.s)) return rc;
  }
  int rc = FMOE_EINVAL;
  switch (x_dtype) {
    case FMOE_F32: rc = launch_fwd_x<float>(a, target_dtype); break;
    case FMOE_BF16: rc = launch_fwd_x<bf16_t>(a, target_dtype); break;
    case FMOE_F16: rc = launch_fwd_x<f16_t>(a, target_dtype); break;
  }
  if (rc || !acc16) return rc;
  return out_dtype == FMOE_BF16
             ? launch_acc_pass<bf16_t>(false, acc, d_out, out_row_stride, hidden, num_tokens, 1,
                                       a.s)
             : launch_acc_pass<f16_t>(false, acc, d_out, out_row_stride, hidden, num_tokens, 1,
                                      a.s);
}

extern "C" int64_t fmoe_combine_det_tile(int64_t num_rows, int64_t num_tokens, int64_t hidden,
                                         int x_dtype) {
  if (num_rows < 1 || num_tokens < 1 || hidden < 1 || !fmoe_host::is_float_dtype(x_dtype)) return -1;
  const int eb = fmoe_host::dtype_bytes(x_dtype);
  if (hidden % (16 / eb) != 0) return 0;
  const fmoe::DetTile c = fmoe::pick_det_tile(num_rows, num_tokens, hidden, eb, 16 / eb);
  int groups = 0;
  for (int g = 2; g <= 4; ++g)
    if (c.lds != 0 && c.lds == fmoe::lds_for_groups(g)) groups = g;
  return groups * 100 + c.U * 10 + c.R;
}

extern "C" int64_t fmoe_combine_small_max_rows(void) { return fmoe::kSmallRows; }

extern "C" int64_t fmoe_combine_atomic_few_groups(int64_t num_rows, int64_t num_tokens,
                                                  int64_t hidden) {
  return fmoe::few_geom(num_rows, num_tokens, hidden).groups;
}

extern "C" int fmoe_combine_fwd_small(const int64_t* host_ptrs, const int64_t* host_rows,
                                      int64_t num_experts, const void* d_indices, int idx_dtype,
                                      const void* d_weights, int w_dtype, int64_t num_tokens,
                                      int64_t hidden, int x_dtype, void* d_out, int out_dtype,
                                      int64_t out_row_stride, int accumulate, int32_t* d_status,
                                      void* stream) {
  using namespace fmoe;
  fmoe_host::clear_error();
  FMOE_REQUIRE(num_tokens >= 1 && hidden >= 1, "fmoe_combine_fwd_small: bad sizes T=%lld D=%lld",
               (long long)num_tokens, (long long)hidden);
  if (num_tokens >= (int64_t(1) << 30) || hidden * 4 >= (int64_t(1) << 31)) {
    fmoe_host::set_error("fmoe_combine_fwd_small: T=%lld / D=%lld exceed the 32-bit counters",
                         (long long)num_tokens, (long long)hidden);
    return FMOE_ERANGE;
  }
  FMOE_REQUIRE(fmoe_host::is_float_dtype(x_dtype), "fmoe_combine_fwd_small: bad x dtype %d",
               x_dtype);
  FMOE_REQUIRE(fmoe_host::is_float_dtype(out_dtype), "fmoe_combine_fwd_small: bad out dtype %d",
               out_dtype);
  FMOE_REQUIRE(fmoe_host::is_index_dtype(idx_dtype), "fmoe_combine_fwd_small: bad index dtype %d",
               idx_dtype);
  FMOE_REQUIRE(fmoe_host::is_float_dtype(w_dtype), "fmoe_combine_fwd_small: bad weight dtype %d",
               w_dtype);
  FMOE_REQUIRE(d_out && d_status, "fmoe_combine_fwd_small: null out / status");
  FMOE_REQUIRE(out_row_stride >= hidden, "fmoe_combine_fwd_small: out row stride %lld < D %lld",
               (long long)out_row_stride, (long long)hidden);
  SmallFwdArgs a{};
  const int64_t xb = x_dtype == FMOE_F32 ? 4 : 2;
  int64_t N = 0;
  if (int rc = small_host_table("fmoe_combine_fwd_small", host_ptrs, host_rows, num_experts,
                                hidden * xb, &a.meta, &N, &a.aligned))
    return rc;
  FMOE_REQUIRE(N == 0 || (d_indices && d_weights), "fmoe_combine_fwd_small: null indices/weights");
  a.idx = d_indices;
  a.idx_dtype = idx_dtype;
  a.w = d_weights;
  a.w_dtype = w_dtype;
  a.N = N;
  a.T = num_tokens;
  a.D = hidden;
  a.out = d_out;
  a.out_stride = out_row_stride;
  a.accumulate = accumulate ? 1 : 0;
  a.status = d_status;
  a.s = static_cast<hipStream_t>(stream);
  switch (x_dtype) {
    case FMOE_F32: return launch_small_x<float>(a, out_dtype);
    case FMOE_BF16: return launch_small_x<bf16_t>(a, out_dtype);
    case FMOE_F16: return launch_small_x<f16_t>(a, out_dtype);
  }
  fmoe_host::set_error("fmoe_combine_fwd_small: bad x dtype %d", x_dtype);
  return FMOE_EINVAL;
}

extern "C" int fmoe_permute_backward(const int32_t* d_slot_pos, int64_t num_tokens, int64_t top_k,
                                     int64_t hidden, int dtype, const void* d_grad_rows,
                                     void* d_grad_x, const void* d_grad_sorted, int gate_dtype,
                                     void* d_grad_gates, void* stream) {
  using namespace fmoe;
  fmoe_host::clear_error();
  const int64_t T = num_tokens, K = top_k, D = hidden;
  FMOE_REQUIRE(T >= 1 && K >= 1 && K <= kWave && D >= 1,
               "fmoe_permute_backward: need T >= 1, D >= 1 and 1 <= top_k <= %d (T=%lld k=%lld "
               "D=%lld)",
               kWave, (long long)T, (long long)K, (long long)D);
  if (T >= (int64_t(1) << 30) || T * K >= (int64_t(1) << 31) || D * 4 >= (int64_t(1) << 31)) {
    fmoe_host::set_error("fmoe_permute_backward: T*k / D exceed the 32-bit counters");
    return FMOE_ERANGE;
  }
  FMOE_REQUIRE(fmoe_host::is_float_dtype(dtype), "fmoe_permute_backward: bad dtype %d", dtype);
  FMOE_REQUIRE(d_slot_pos && d_grad_rows && d_grad_x, "fmoe_permute_backward: null device pointer");
  FMOE_REQUIRE((d_grad_sorted == nullptr) == (d_grad_gates == nullptr),
               "fmoe_permute_backward: gate gradients need both pointers, or neither");
  FMOE_REQUIRE(!d_grad_gates || fmoe_host::is_float_dtype(gate_dtype),
               "fmoe_permute_backward: bad gate dtype %d", gate_dtype);
  const SlotsBwdArgs a{d_slot_pos, T, K, D, d_grad_rows, d_grad_x, d_grad_sorted, d_grad_gates,
                       static_cast<hipStream_t>(stream), 0};
  switch (dtype) {
    case FMOE_F32: return launch_slots_bwd<float>(a, gate_dtype);
    case FMOE_BF16: return launch_slots_bwd<bf16_t>(a, gate_dtype);
    default: return launch_slots_bwd<f16_t>(a, gate_dtype);
  }
}
