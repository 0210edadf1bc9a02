// feat3amd_transpose.hip -- the transposed CSR apply of Arch::Apply::csr in a fixed order.
//
// The reference's generic transposed apply (arch/apply_generic.hpp:37-53) is
//     r = (b/a) * (|b| < eps ? 0 : y);   r[col[i]] += val[i] * x[row];   r = a * r
// with the scatter running over the rows in order, so every r[c] accumulates its
// column's entries in ascending entry order.  Here each call collects the entries of every
// column (entries counted per column, the counts summed up, entry and row number written to
// the column's place), sorts each column's short list by entry number and adds it up in that
// order: the same additions in the same order, with no atomics on values, so the result is
// deterministic and bit-identical to the sequential loop.
//
// A stable radix sort of all entries by column, with one lane per column following the sorted
// entries one dependent load at a time, took 0.68 ms on 7.1 M entries (3D Q1 level 6), 0.35 ms
// of it the gather; the lists cost one pass of counting atomics (119 us, the largest part now)
// and one of placing (67 us) instead of three sort passes, and a workgroup loads all entries of
// its 32 columns at once (63 us): 0.32 ms in all.  Dense columns gain most (64 of 100,000 entries
// 41 -> 4.4 ms, 300 of 30,000 22 -> 1.6 ms, 4000 of 1100 1.4 -> 0.74 ms).  Where the columns of a
// large matrix are entirely random the sort was better, as every counting atomic and every placed
// word is a cache line of its own: 6 M entries in 300 k columns 0.61 -> 0.52 ms, 5 M in 50 k columns
// 0.41 -> 0.52, 20 M in 1 M columns 2.0 -> 2.3, 20 M in 150 k columns 2.0 -> 2.3 ms.
//
// The buffers of the allocating form come stream-ordered from a pool of the handle's own, which
// keeps up to kTrPoolBytes between calls (the device's default pool gives everything back at
// every synchronisation: 2.3 ms for a call that is waited for, 0.42 ms now); the
// allocation-free variant keeps them in a static device array instead.
#include "feat3amd_common.hpp"

#include <algorithm>
#include <mutex>

// Scratch of the allocation-free variant (feat_csr_apply_transposed_noalloc_f64_u64): the
// column lists live in this file-scope device array, one copy per GPU, held until the
// process ends.  Host code never passes `scratch` itself to a kernel or copy (on the host
// the name is only a stand-in for the symbol): it uses the per-device address that
// hipGetSymbolAddress returned at handle creation.  Every call on one GPU shares that
// GPU's copy, so calls that overlap on one GPU race; nothing in it needs to start at zero.
// Beyond the documented size it holds what does not grow with the entries: the scan's sums (4
// bytes for each kTrScan columns) and the alignment of the parts.
constexpr size_t kTrScratchSlack = size_t(64) << 10;
static __device__ __align__(256) unsigned char scratch[FEAT_TR_NOALLOC_SCRATCH_BYTES + kTrScratchSlack];

namespace {

constexpr size_t kTrScratchBytes = size_t(FEAT_TR_NOALLOC_SCRATCH_BYTES);
constexpr uint64_t kTrPoolBytes = uint64_t(256) << 20;   // most a handle keeps between calls
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

void* scratch_of(int device)
{
  if(device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mutex);
  return g_scratch_ptr[device];
}

constexpr uint32_t kTrScan = 1024;     // counts a workgroup scans
constexpr uint32_t kTrTile = 4096;     // entries a workgroup places
constexpr uint32_t kTrCols = 32;       // columns a workgroup adds up
constexpr uint32_t kTrPer = kThreads / kTrCols;   // threads a column
constexpr uint32_t kTrCap = 1024;      // entries it holds in LDS at a time (27-point rows: 864)
constexpr uint32_t kTrShort = 192;     // longest list that shares a workgroup
constexpr uint32_t kTrParts = 1024;    // parts by entry number that a longer list is split into at a time
constexpr uint32_t kTrWindow = 262144; // most entries that are split into parts at a time
constexpr uint32_t kTrSpread = 512;    // fewest workgroups while there may be long lists

__global__ void k_tr_zero(uint32_t* p, uint64_t n)
{
  for(uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x) p[i] = 0;
}

// cnt[c]: entries of column c; rank[e]: a number of its own for entry e within its column
template<typename IT>
__global__ __launch_bounds__(kThreads) void k_tr_count(const IT* __restrict__ col, uint64_t nnz, uint32_t* cnt,
                                                       uint32_t* __restrict__ rank)
{
  const uint64_t stride = uint64_t(gridDim.x) * kThreads;
  for(uint64_t e0 = blockIdx.x * uint64_t(kThreads) + threadIdx.x; e0 < nnz; e0 += 4 * stride)
  {
    IT c[4];
    uint32_t k[4];
#pragma unroll
    for(int u = 0; u < 4; ++u) c[u] = e0 + u * stride < nnz ? col[e0 + u * stride] : IT(0);
#pragma unroll
    for(int u = 0; u < 4; ++u) k[u] = e0 + u * stride < nnz ? atomicAdd(cnt + c[u], 1u) : 0u;
#pragma unroll
    for(int u = 0; u < 4; ++u)
      if(e0 + u * stride < nnz) rank[e0 + u * stride] = k[u];
  }
}

// exclusive sum over the workgroup's kThreads values
__device__ uint32_t block_scan(uint32_t v, uint32_t* sh /* kThreads / 64 */, uint32_t& total)
{
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t s = v;
  for(int d = 1; d < 64; d <<= 1)
  {
    const uint32_t t = __shfl_up(s, d, 64);
    if(lane >= d) s += t;
  }
  if(lane == 63) sh[w] = s;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
  for(int i = 0; i < kThreads / 64; ++i)
  {
    if(i < w) before += sh[i];
    total += sh[i];
  }
  __syncthreads();
  return before + s - v;
}

__global__ __launch_bounds__(kThreads) void k_tr_sums(const uint32_t* cnt, uint64_t n, uint32_t* sums)
{
  __shared__ uint32_t sh[kThreads / 64];
  uint32_t v = 0, total;
  for(uint32_t u = 0; u < kTrScan / kThreads; ++u)
  {
    const uint64_t i = uint64_t(blockIdx.x) * kTrScan + u * kThreads + threadIdx.x;
    if(i < n) v += cnt[i];
  }
  (void)block_scan(v, sh, total);
  if(threadIdx.x == 0) sums[blockIdx.x] = total;
}

// exclusive sums of the nb workgroup sums, in place (one workgroup)
__global__ __launch_bounds__(kThreads) void k_tr_scan_sums(uint32_t* sums, uint32_t nb)
{
  __shared__ uint32_t sh[kThreads / 64];
  uint32_t carry = 0;
  for(uint32_t i0 = 0; i0 < nb; i0 += kThreads)
  {
    const uint32_t i = i0 + threadIdx.x;
    uint32_t total;
    const uint32_t s = block_scan(i < nb ? sums[i] : 0u, sh, total);
    if(i < nb) sums[i] = carry + s;
    carry += total;
  }
}

// counts -> first positions, in place; ptr[n] = all entries.  The columns of more than kTrShort
// entries go to longs[0 .. ptr[n + 1]), in any order.
__global__ __launch_bounds__(kThreads) void k_tr_colptr(uint32_t* ptr, uint64_t n, const uint32_t* sums, uint32_t nnz,
                                                        uint32_t* longs)
{
  __shared__ uint32_t sh[kThreads / 64];
  uint32_t carry = sums[blockIdx.x];
  for(uint32_t u = 0; u < kTrScan / kThreads; ++u)
  {
    const uint64_t i = uint64_t(blockIdx.x) * kTrScan + u * kThreads + threadIdx.x;
    uint32_t total;
    const uint32_t v = i < n ? ptr[i] : 0u;
    const uint32_t s = block_scan(v, sh, total);
    if(i < n) ptr[i] = carry + s;
    carry += total;
    const uint64_t lng = __ballot(v > kTrShort);
    if(lng)
    {
      const int lane = threadIdx.x & 63, first = __ffsll((unsigned long long)lng) - 1;
      uint32_t at = 0;
      if(lane == first) at = atomicAdd(ptr + n + 1, uint32_t(__popcll(lng)));
      at = __shfl(at, first, 64);
      if(v > kTrShort) longs[at + uint32_t(__popcll(lng & ((uint64_t(1) << lane) - 1)))] = uint32_t(i);
    }
  }
  if(blockIdx.x == 0 && threadIdx.x == 0) ptr[n] = nnz;
}

// list[position] = entry number (high half) and row (low half): ascending words = ascending entries
template<typename IT>
__global__ __launch_bounds__(kThreads) void k_tr_place(const IT* __restrict__ col, const IT* __restrict__ rowptr,
                                                       uint64_t rows, uint64_t nnz, const uint32_t* __restrict__ colptr,
                                                       const uint32_t* __restrict__ rank, uint64_t* __restrict__ list)
{
  __shared__ uint32_t srp[kTrTile + 2];
  __shared__ uint64_t sr[2];
  for(uint64_t e0 = uint64_t(blockIdx.x) * kTrTile; e0 < nnz; e0 += uint64_t(gridDim.x) * kTrTile)
  {
    const uint64_t e1 = e0 + kTrTile < nnz ? e0 + kTrTile : nnz;
    // the rows of the tile's first and last entry: the last r with rowptr[r] <= e
    if(threadIdx.x < 2)
    {
      const uint64_t e = threadIdx.x ? e1 - 1 : e0;
      uint64_t lo = 0, hi = rows;
      while(hi - lo > 1)
      {
        const uint64_t mid = (lo + hi) >> 1;
        if(uint64_t(rowptr[mid]) <= e)
          lo = mid;
        else
          hi = mid;
      }
      sr[threadIdx.x] = lo;
    }
    __syncthreads();
    const uint64_t r0 = sr[0], nr = sr[1] - sr[0] + 1;
    const bool in_lds = nr <= kTrTile + 1;
    if(in_lds)
      for(uint64_t i = threadIdx.x; i < nr; i += kThreads) srp[i] = uint32_t(rowptr[r0 + i]);
    __syncthreads();
    for(uint64_t e = e0 + threadIdx.x; e < e1; e += kThreads)
    {
      const uint64_t c = uint64_t(col[e]);
      const uint32_t k = rank[e];
      uint64_t lo = 0, hi = nr;
      while(hi - lo > 1)
      {
        const uint64_t mid = (lo + hi) >> 1;
        const uint64_t v = in_lds ? uint64_t(srp[mid]) : uint64_t(rowptr[r0 + mid]);
        if(v <= e)
          lo = mid;
        else
          hi = mid;
      }
      list[colptr[c] + k] = (e << 32) | (r0 + lo);
    }
    __syncthreads();
  }
}

// ascending sort of a[0 .. n) by the whole workgroup (bitonic network; pairs with one end at or
// beyond n are already in order, as if the missing words were larger than all)
__device__ void block_sort(uint64_t* a, uint32_t n)
{
  uint32_t p = 2;
  for(; p < 2 * n && p; p <<= 1)
  {
    // first step of a merge: mirrored pairs, the further ones at distance d
    for(uint32_t i = threadIdx.x; i < (n + p - 1) / p * (p / 2); i += kThreads)
    {
      const uint32_t b = i / (p / 2) * p, o = i % (p / 2), l = b + o, h = b + p - 1 - o;
      if(h < n)
      {
        const uint64_t x = a[l], y = a[h];
        if(y < x)
        {
          a[l] = y;
          a[h] = x;
        }
      }
    }
    __syncthreads();
    for(uint32_t d = p / 4; d; d >>= 1)
    {
      for(uint32_t i = threadIdx.x; i < (n + 2 * d - 1) / (2 * d) * d; i += kThreads)
      {
        const uint32_t l = i / d * 2 * d + i % d, h = l + d;
        if(h < n)
        {
          const uint64_t x = a[l], y = a[h];
          if(y < x)
          {
            a[l] = y;
            a[h] = x;
          }
        }
      }
      __syncthreads();
    }
  }
}

// per <= kTrCols columns a workgroup, kTrPer threads a column.  A thread holds up to 4 entries of its
// column's list at a time and counts the smaller entry numbers in it, while the entries' values
// and x are on their way; both go to their place in LDS, and one lane a column adds them in
// order.  (One lane a column sorting its list in LDS took 233 us instead of 63.)
//
// Columns of more than kTrShort entries are left to the end, one workgroup each, whichever columns
// they are (32 neighbours one after the other in the workgroup of their group: 64 columns of
// 100,000 entries 300 ms, 64 of 1000 entries 1.1 ms, now 4.4 and 0.08).  A list is split by entry number
// into kTrParts parts (counted, then written part by part: in LDS up to kTrCap entries, else to
// `spare`), and an entry's place is its part's begin and its rank in its part.  A part of more
// than kTrCap entries is sorted where it lies; lists beyond kTrWindow entries are split a window of
// entry numbers at a time, so that evenly spread parts fit.
template<typename DT>
__global__ __launch_bounds__(kThreads) void k_tr_gather(DT* r, DT a, DT ba, const DT* x, const DT* y, int bzero,
                                                        const DT* val, const uint32_t* colptr, const uint64_t* list,
                                                        const uint32_t* longs, uint64_t* spare, uint64_t cols, uint32_t per)
{
  __shared__ uint32_t se[kTrCap], part[kTrParts];
  __shared__ DT sv[kTrCap], sx[kTrCap];
  __shared__ uint32_t cp[kTrCols + 1], sh[kThreads / 64], lim[2];
  const uint32_t t = threadIdx.x, tc = t / kTrPer, sub = t % kTrPer;
  for(uint64_t c0 = uint64_t(blockIdx.x) * per; c0 < cols; c0 += uint64_t(gridDim.x) * per)
  {
    const uint32_t nc = cols - c0 < per ? uint32_t(cols - c0) : per;
    if(t <= nc) cp[t] = colptr[c0 + t];
    __syncthreads();
    for(uint32_t c = 0; c < nc;)
    {
      // the next columns that fit together, or one long column (left out)
      const uint32_t p0 = cp[c];
      const bool lng = cp[c + 1] - p0 > kTrShort;
      uint32_t ce = c + 1;
      if(!lng)
        while(ce < nc && cp[ce + 1] - p0 <= kTrCap && cp[ce + 1] - cp[ce] <= kTrShort) ++ce;
      if(!lng)
      {
        DT acc = DT(0);
        if(t < ce - c) acc = ba * (bzero ? DT(0) : y[c0 + c + t]);
        const bool on = tc < ce - c;
        const uint32_t b = on ? cp[c + tc] - p0 : 0, e = on ? cp[c + tc + 1] - p0 : 0;
        for(uint32_t i = b + sub; i < e; i += kTrPer) se[i] = uint32_t(list[p0 + i] >> 32);
        __syncthreads();
        for(uint32_t i0 = b + sub; i0 < e; i0 += 4 * kTrPer)
        {
          uint32_t en[4], rank[4];
          DT v[4], xv[4];
#pragma unroll
          for(uint32_t u = 0; u < 4; ++u)
          {
            const uint32_t i = i0 + u * kTrPer;
            const uint64_t w = i < e ? list[p0 + i] : list[p0 + i0];
            en[u] = uint32_t(w >> 32);
            v[u] = val[w >> 32];
            xv[u] = x[uint32_t(w)];
            rank[u] = 0;
          }
#pragma unroll 4
          for(uint32_t j = b; j < e; ++j)
          {
            const uint32_t o = se[j];
#pragma unroll
            for(uint32_t u = 0; u < 4; ++u) rank[u] += o < en[u] ? 1u : 0u;
          }
#pragma unroll
          for(uint32_t u = 0; u < 4; ++u)
            if(i0 + u * kTrPer < e)
            {
              sv[b + rank[u]] = v[u];
              sx[b + rank[u]] = xv[u];
            }
        }
        __syncthreads();
        if(t < ce - c)
        {
          const uint32_t bt = cp[c + t] - p0, et = cp[c + t + 1] - p0;
#pragma unroll 4
          for(uint32_t i = bt; i < et; ++i) acc = dfma(sv[i], sx[i], acc);
          r[c0 + c + t] = a * acc;
        }
        __syncthreads();
      }
      c = ce;
    }
    __syncthreads();   // cp
  }
  const uint32_t nlong = colptr[cols + 1];
  for(uint32_t l = blockIdx.x; l < nlong; l += gridDim.x)
  {
    const uint32_t c = longs[l], p0 = colptr[c], n = colptr[c + 1] - p0;
    DT acc = DT(0);
    if(t == 0) acc = ba * (bzero ? DT(0) : y[c]);
    // adds sv[i] sx[i], i < m, in order
    auto sum = [&](uint32_t m) {
      __syncthreads();
      if(t == 0)
      {
#pragma unroll 4
        for(uint32_t i = 0; i < m; ++i) acc = dfma(sv[i], sx[i], acc);
      }
      __syncthreads();
    };
    // exclusive sums of part[], from carry on; the total with it
    auto scan = [&](uint32_t carry) -> uint32_t {
      uint32_t v[kTrParts / kThreads], own = 0, total;
      for(uint32_t u = 0; u < kTrParts / kThreads; ++u) own += v[u] = part[t * (kTrParts / kThreads) + u];
      uint32_t at = carry + block_scan(own, sh, total);
      for(uint32_t u = 0; u < kTrParts / kThreads; ++u)
      {
        part[t * (kTrParts / kThreads) + u] = at;
        at += v[u];
      }
      __syncthreads();
      return carry + total;
    };
    const uint64_t* src = list + p0;
    // f(word) for the thread's words of the list, eight loads in flight
    auto each = [&](auto f) {
      for(uint32_t i0 = t; i0 < n; i0 += 8 * kThreads)
      {
        uint64_t w[8];
#pragma unroll
        for(uint32_t u = 0; u < 8; ++u) w[u] = src[i0 + u * kThreads < n ? i0 + u * kThreads : i0];
#pragma unroll
        for(uint32_t u = 0; u < 8; ++u)
          if(i0 + u * kThreads < n) f(w[u]);
      }
    };
    constexpr uint32_t kOwn = kTrCap / kThreads;
    // the m <= kTrCap words at from, se[] holding their entry numbers in the order of their parts
    // (part k: se[end of part k - 1 .. part[k]), both less b): values and x to their places
    auto place_in_parts = [&](const uint64_t (&w)[kOwn], uint32_t m, uint32_t base, uint32_t shift, uint32_t b) {
      DT v[kOwn], xv[kOwn];
#pragma unroll
      for(uint32_t u = 0; u < kOwn; ++u)
        if(t + u * kThreads < m)
        {
          v[u] = val[w[u] >> 32];
          xv[u] = x[uint32_t(w[u])];
        }
#pragma unroll
      for(uint32_t u = 0; u < kOwn; ++u)
        if(t + u * kThreads < m)
        {
          const uint32_t e = uint32_t(w[u] >> 32), k = ((e - base) >> shift) % kTrParts;
          const uint32_t kb = k && part[k - 1] > b ? part[k - 1] - b : 0, ke = part[k] - b;
          uint32_t rank = kb;
#pragma unroll 8
          for(uint32_t q = kb; q < ke; ++q) rank += se[q] < e ? 1u : 0u;
          sv[rank] = v[u];
          sx[rank] = xv[u];
        }
    };
    if(t < 2) lim[t] = t ? 0u : ~0u;
    for(uint32_t i = t; i < kTrParts; i += kThreads) part[i] = 0;
    __syncthreads();
    uint32_t lo = ~0u, hi = 0;
    each([&](uint64_t w) {
      const uint32_t e = uint32_t(w >> 32);
      lo = e < lo ? e : lo;
      hi = e > hi ? e : hi;
    });
    atomicMin(&lim[0], lo);
    atomicMax(&lim[1], hi);
    __syncthreads();
    // 2^wbits windows of kTrParts = 2^10 parts of 2^shift entry numbers each
    const uint32_t first = lim[0], bits = 32 - uint32_t(__clz(int(lim[1] - first)));
    if(n <= kTrCap)
    {
      const uint32_t shift = bits > 10 ? bits - 10 : 0;
      uint64_t w[kOwn];
#pragma unroll
      for(uint32_t u = 0; u < kOwn; ++u)
      {
        w[u] = t + u * kThreads < n ? src[t + u * kThreads] : 0;
        if(t + u * kThreads < n) atomicAdd(&part[(uint32_t(w[u] >> 32) - first) >> shift], 1u);
      }
      __syncthreads();
      (void)scan(0);
#pragma unroll
      for(uint32_t u = 0; u < kOwn; ++u)
        if(t + u * kThreads < n)
        {
          const uint32_t e = uint32_t(w[u] >> 32);
          se[atomicAdd(&part[(e - first) >> shift], 1u)] = e;
        }
      __syncthreads();   // part[k]: now the end of part k
      place_in_parts(w, n, first, shift, 0);
      sum(n);
    }
    else
    {
      uint64_t* dst = spare + p0;
      uint32_t wbits = 0;
      while((n >> wbits) > kTrWindow) ++wbits;
      const uint32_t shift = bits - 10 - wbits;   // n > 2^(10 + wbits) different numbers
      uint32_t done = 0;                          // entries of the windows before
      for(uint32_t win = 0; win < (1u << wbits); ++win)
      {
        each([&](uint64_t w) {
          const uint32_t k = (uint32_t(w >> 32) - first) >> shift;
          if(k / kTrParts == win) atomicAdd(&part[k % kTrParts], 1u);
        });
        __syncthreads();
        const uint32_t all = scan(done);
        each([&](uint64_t w) {
          const uint32_t k = (uint32_t(w >> 32) - first) >> shift;
          if(k / kTrParts == win) dst[atomicAdd(&part[k % kTrParts], 1u)] = w;
        });
        __syncthreads();   // part[k]: now the end of part k
        for(uint32_t k = 0, b = done; k < kTrParts;)
        {
          uint32_t e = part[k++];
          while(k < kTrParts && part[k] - b <= kTrCap) e = part[k++];
          if(e - b <= kTrCap)
          {
            uint64_t w[kOwn];
#pragma unroll
            for(uint32_t u = 0; u < kOwn; ++u)
            {
              const uint32_t i = t + u * kThreads;
              w[u] = b + i < e ? dst[b + i] : 0;
              if(b + i < e) se[i] = uint32_t(w[u] >> 32);
            }
            __syncthreads();
            place_in_parts(w, e - b, first, shift, b);
            sum(e - b);
          }
          else
          {
            block_sort(dst + b, e - b);
            for(uint32_t q = b; q < e; q += kTrCap)
            {
              const uint32_t m = e - q < kTrCap ? e - q : kTrCap;
              for(uint32_t i = t; i < m; i += kThreads)
              {
                const uint64_t w = dst[q + i];
                sv[i] = val[w >> 32];
                sx[i] = x[uint32_t(w)];
              }
              sum(m);
            }
          }
          b = e;
        }
        done = all;
        __syncthreads();
        for(uint32_t i = t; i < kTrParts; i += kThreads) part[i] = 0;
        __syncthreads();
      }
    }
    if(t == 0) r[c] = a * acc;
  }
}

// 256-byte aligned bump layout inside one buffer
struct ScratchLayout
{
  size_t off = 0;
  template<typename T>
  size_t take(uint64_t n)
  {
    const size_t o = off;
    off = (off + sizeof(T) * size_t(n ? n : 1) + 255) & ~size_t(255);
    return o;
  }
};

struct TrLayout
{
  size_t colptr, sums, longs, spare, list, bytes;
  uint32_t nb;
  TrLayout(uint64_t cols, uint64_t nnz) : nb(uint32_t((cols + kTrScan - 1) / kTrScan))
  {
    ScratchLayout lay;
    colptr = lay.take<uint32_t>(cols + 2);   // and the number of long columns
    sums = lay.take<uint32_t>(nnz ? nb : 0);
    longs = lay.take<uint32_t>(nnz / (kTrShort + 1));
    spare = lay.take<uint64_t>(nnz);   // the ranks until the lists are written
    list = lay.take<uint64_t>(nnz);
    bytes = lay.off;
  }
};

// the transposed apply with its buffers at base (cols > 0)
template<typename DT, typename IT>
int tr_apply(hipStream_t s, unsigned char* base, const TrLayout& L, DT* r, DT a, const DT* x, DT b, bool bzero, const DT* y,
             const DT* val, const IT* col, const IT* rowptr, uint64_t rows, uint64_t cols, uint64_t nnz, const char* name)
{
  uint32_t* colptr = reinterpret_cast<uint32_t*>(base + L.colptr);
  uint32_t* sums = reinterpret_cast<uint32_t*>(base + L.sums);
  uint32_t* longs = reinterpret_cast<uint32_t*>(base + L.longs);
  uint64_t* spare = reinterpret_cast<uint64_t*>(base + L.spare);
  uint32_t* rank = reinterpret_cast<uint32_t*>(spare);
  uint64_t* list = reinterpret_cast<uint64_t*>(base + L.list);
  hipLaunchKernelGGL(k_tr_zero, dim3(grid_for(cols + 2)), dim3(kThreads), 0, s, colptr, cols + 2);
  if(nnz)
  {
    hipLaunchKernelGGL((k_tr_count<IT>), dim3(grid_for(nnz, 4)), dim3(kThreads), 0, s, col, nnz, colptr, rank);
    hipLaunchKernelGGL(k_tr_sums, dim3(L.nb), dim3(kThreads), 0, s, colptr, cols, sums);
    hipLaunchKernelGGL(k_tr_scan_sums, dim3(1), dim3(kThreads), 0, s, sums, L.nb);
    hipLaunchKernelGGL(k_tr_colptr, dim3(L.nb), dim3(kThreads), 0, s, colptr, cols, sums, uint32_t(nnz), longs);
    const uint64_t tiles = (nnz + kTrTile - 1) / kTrTile;
    hipLaunchKernelGGL((k_tr_place<IT>), dim3(unsigned(std::min<uint64_t>(tiles, kMaxGrid))), dim3(kThreads), 0, s, col,
                       rowptr, rows, nnz, colptr, rank, list);
  }
  // kTrCols columns a workgroup, fewer where that leaves the chip idle
  const uint64_t per = std::min<uint64_t>(std::max<uint64_t>(cols / kTrSpread, 4), kTrCols);
  const uint64_t groups = std::max((cols + per - 1) / per, std::min<uint64_t>(nnz / (kTrShort + 1), kTrSpread));
  hipLaunchKernelGGL((k_tr_gather<DT>), dim3(unsigned(std::min<uint64_t>(groups, kMaxGrid))), dim3(kThreads), 0, s, r, a,
                     DT(b / a), x, y, int(bzero), val, colptr, list, longs, spare, cols, uint32_t(per));
  return check_launch(name);
}

} // namespace

namespace feat3amd_detail {

int noalloc_scratch_attach(int device)
{
  if(device < 0 || device >= kMaxDevices) return fail(FEAT_ERR_UNSUPPORTED, "no-alloc scratch: device index above 63");
  std::lock_guard<std::mutex> lk(g_scratch_mutex);
  if(g_scratch_ptr[device]) return FEAT_OK;
  void* p = nullptr;
  const int rc = check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
  if(rc) return rc;
  g_scratch_ptr[device] = p;
  return FEAT_OK;
}

// The transposed apply of csr_apply_transposed with every buffer in the device's scratch
// array: no allocation, no free; sizes that do not fit are rejected before any launch.
template<typename DT, typename IT>
int csr_apply_transposed_noalloc(feat_handle_t h, DT* r, DT a, const DT* x, DT b, bool bzero, const DT* y,
                                 const DT* val, const IT* col, const IT* rowptr, uint64_t rows, uint64_t cols,
                                 uint64_t nnz, const char* name)
{
  if(nnz >= (uint64_t(1) << 31) || rows >= (uint64_t(1) << 32) || cols >= (uint64_t(1) << 32))
    return fail(FEAT_ERR_UNSUPPORTED, "csr_apply_transposed_noalloc: needs fewer than 2^31 entries and 2^32 rows, columns");
  unsigned char* base = static_cast<unsigned char*>(scratch_of(h->device));
  if(!base) return fail(FEAT_ERR_NO_DEVICE, "csr_apply_transposed_noalloc: scratch not attached on the handle's device");
  if(!cols) return FEAT_OK;
  // the documented limit, 20 bytes per entry and 4 per column, is wider than the lists' 16 and 4
  if(20 * nnz + 4 * cols > kTrScratchBytes)
    return fail(FEAT_ERR_UNSUPPORTED, "csr_apply_transposed_noalloc: the matrix needs more than the 32 MiB scratch "
                                      "(20 bytes per entry and 4 per column)");
  const TrLayout L(cols, nnz);
  if(L.bytes > kTrScratchBytes + kTrScratchSlack)
    return fail(FEAT_ERR_UNSUPPORTED, "csr_apply_transposed_noalloc: the matrix needs more than the 32 MiB scratch");
  return tr_apply(h->stream, base, L, r, a, x, b, bzero, y, val, col, rowptr, rows, cols, nnz, name);
}

template int csr_apply_transposed_noalloc<double, uint64_t>(feat_handle_t, double*, double, const double*, double, bool,
                                                            const double*, const double*, const uint64_t*,
                                                            const uint64_t*, uint64_t, uint64_t, uint64_t, const char*);

// the handle's pool, made at its first use
static int pool_of(feat_handle_t h, hipMemPool_t* pool)
{
  std::lock_guard<std::mutex> lk(h->pool_mutex);
  if(!h->pool)
  {
    hipMemPoolProps props = {};
    props.allocType = hipMemAllocationTypePinned;
    props.handleTypes = hipMemHandleTypeNone;
    props.location.type = hipMemLocationTypeDevice;
    props.location.id = h->device;
    hipMemPool_t p = nullptr;
    int rc = check_hip(hipMemPoolCreate(&p, &props), "transposed apply: pool");
    if(rc) return rc;
    uint64_t keep = kTrPoolBytes;
    rc = check_hip(hipMemPoolSetAttribute(p, hipMemPoolAttrReleaseThreshold, &keep), "transposed apply: pool");
    if(rc)
    {
      (void)hipMemPoolDestroy(p);
      return rc;
    }
    h->pool = p;
  }
  *pool = h->pool;
  return FEAT_OK;
}

template<typename DT, typename IT>
int csr_apply_transposed(feat_handle_t h, DT* r, DT a, const DT* x, DT b, bool bzero, const DT* y, const DT* val,
                         const IT* col, const IT* rowptr, uint64_t rows, uint64_t cols, uint64_t nnz, const char* name)
{
  if(nnz >= (uint64_t(1) << 31) || rows >= (uint64_t(1) << 32) || cols >= (uint64_t(1) << 32))
    return fail(FEAT_ERR_UNSUPPORTED, "csr_apply: transposed apply needs fewer than 2^31 entries and 2^32 rows, columns");
  if(!cols) return FEAT_OK;
  const TrLayout L(cols, nnz);
  hipMemPool_t pool = nullptr;
  void* base = nullptr;
  int rc = pool_of(h, &pool);
  if(!rc) rc = check_hip(hipMallocFromPoolAsync(&base, L.bytes, pool, h->stream), "transposed apply: buffer");
  if(rc) return rc;
  rc = tr_apply(h->stream, static_cast<unsigned char*>(base), L, r, a, x, b, bzero, y, val, col, rowptr, rows, cols, nnz, name);
  (void)hipFreeAsync(base, h->stream);
  return rc;
}

template int csr_apply_transposed<double, uint64_t>(feat_handle_t, double*, double, const double*, double, bool,
                                                    const double*, const double*, const uint64_t*, const uint64_t*,
                                                    uint64_t, uint64_t, uint64_t, const char*);
template int csr_apply_transposed<double, uint32_t>(feat_handle_t, double*, double, const double*, double, bool,
                                                    const double*, const double*, const uint32_t*, const uint32_t*,
                                                    uint64_t, uint64_t, uint64_t, const char*);
template int csr_apply_transposed<float, uint64_t>(feat_handle_t, float*, float, const float*, float, bool,
                                                   const float*, const float*, const uint64_t*, const uint64_t*,
                                                   uint64_t, uint64_t, uint64_t, const char*);
template int csr_apply_transposed<float, uint32_t>(feat_handle_t, float*, float, const float*, float, bool,
                                                   const float*, const float*, const uint32_t*, const uint32_t*,
                                                   uint64_t, uint64_t, uint64_t, const char*);

} // namespace feat3amd_detail
