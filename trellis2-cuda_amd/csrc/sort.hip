// Stable LSD radix argsort of 27-bit keys: 3 passes of 9-bit digits. It produces the reference's `sorted`
// permutation (src/spconv.cu:47-52: cub::DeviceRadixSort::SortPairs(bin -> iota), stable, bits 0..32; bin < 2^27
// so bits 27..31 are all zero and sorting 27 bits gives the same order).
//
// Up to kSmallKeys keys: one launch per pass (k_rs_pass).
// More: three launches per pass over tiles of 256 x RCH keys (RCH = 4, 8 or 16, so there are at least ~900 tiles when
// the input allows it):
//   count      : per-tile digit counts, tile-major [ntiles][512], so that a tile's counts are whole lines (the first
//                one also zeroes the digit-sum slots; a producer that already holds the keys may count the first pass
//                itself, see SortWork)
//   digit scan : one workgroup per 16 digits sums their columns and publishes the sums; a digit's start is the sum of
//                the lower digits' published sums (read back all at once); the columns become exclusive tile starts.
//                One launch instead of a device-wide scan's three.
//   scatter    : each wavefront ranks its chunks of 64 keys in order; within a chunk, lanes holding the same digit
//                find each other with 9 ballots (one per digit bit) and take rank = popcount(peers below me);
//                wavefront counts are prefixed across the 4 wavefronts. Destination = tile start + wavefronts
//                before + rank, so every key keeps its input order among equal digits.
// Measured against a look-back (single-pass) form with tile tickets: the per-digit look-back chains cost more than
// the two extra launches at every size here (C3 build 0.128 -> 0.106 ms, C4 0.400 -> 0.382 ms).
#include "scan.h"

namespace {
constexpr int RBITS = 9, NBUK = 1 << RBITS, RT = 256;
constexpr uint64_t ST_SUM = 1ull << 32;  // published flag of a digit-sum slot
constexpr uint32_t kSpinLimit = 1u << 20;  // default bound of the digit-sum wait (SPCONV_SORT_SPIN_LIMIT)

// Ranks a wavefront's RCH chunks of 64 keys (rows seg .. seg + RCH*64) by the digit at `shift`, in input order: lanes
// holding the same digit find each other with RBITS ballots and take rank = popcount(peers below me) plus the
// wavefront's running count for that digit (cw, in LDS, zeroed by the caller), which the lowest peer advances.
template <int RCH>
__device__ __forceinline__ void rank_chunks(const uint32_t* __restrict__ kin, const int32_t* __restrict__ vin, i64 n,
                                            int shift, i64 seg, int lane, uint32_t* cw, uint32_t (&key)[RCH],
                                            int32_t (&val)[RCH], uint32_t (&rank)[RCH]) {
  const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll
  for (int c = 0; c < RCH; c++) {
    const i64 i = seg + c * 64 + lane;
    const bool ok = i < n;
    key[c] = ok ? kin[i] : 0u;
    val[c] = ok ? (vin ? vin[i] : (int32_t)i) : 0;
    const uint32_t d = (key[c] >> shift) & (NBUK - 1);
    uint64_t peers = __ballot(ok);
#pragma unroll
    for (int b = 0; b < RBITS; b++) {
      const uint64_t m = __ballot((d >> b) & 1u);
      peers &= ((d >> b) & 1u) ? m : ~m;
    }
    const uint32_t r = (uint32_t)__popcll(peers & lt);
    const uint32_t before = ok ? cw[d] : 0u;
    rank[c] = before + r;
    if (ok && r == 0) cw[d] = before + (uint32_t)__popcll(peers);
  }
}

// Per-tile digit counts. Workgroup 0 also zeroes `zero` (zn words: the digit-sum slots of every pass, before the
// first digit scan reads them), which saves the sort a launch.
template <int RCH>
__global__ void __launch_bounds__(RT) k_rs_count(const uint32_t* __restrict__ keys, i64 n, int shift,
                                                 uint32_t* __restrict__ hist, uint32_t* __restrict__ zero,
                                                 int zn, const uint32_t* __restrict__ ndev) {
  __shared__ uint32_t cnt[NBUK];
  if (ndev) {  // device-side key count: tiles past it are skipped (the digit scan reads only the tiles below it)
    n = min<i64>(n, *ndev);
    if (blockIdx.x > 0 && (i64)blockIdx.x * (RT * RCH) >= n) return;
  }
  if (zero && blockIdx.x == 0)
    for (int i = threadIdx.x; i < zn; i += RT) zero[i] = 0;
  for (int d = threadIdx.x; d < NBUK; d += RT) cnt[d] = 0;
  __syncthreads();
  i64 base = (i64)blockIdx.x * (RT * RCH);
#pragma unroll 4
  for (int j = 0; j < RCH; j++) {
    i64 i = base + j * RT + threadIdx.x;
    if (i < n) atomicAdd(&cnt[(keys[i] >> shift) & (NBUK - 1)], 1u);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < NBUK; d += RT) hist[(i64)blockIdx.x * NBUK + d] = cnt[d];
}

template <int RCH>
__global__ void __launch_bounds__(RT) k_rs_scatter(const uint32_t* __restrict__ kin, const int32_t* __restrict__ vin,
                                                   uint32_t* __restrict__ kout, int32_t* __restrict__ vout, i64 n,
                                                   int shift, const uint32_t* __restrict__ start,
                                                   const uint32_t* __restrict__ ndev) {
  __shared__ uint32_t cnt[RT / 64][NBUK];
  if (ndev) {
    n = min<i64>(n, *ndev);
    if (blockIdx.x > 0 && (i64)blockIdx.x * (RT * RCH) >= n) return;  // no keys in this tile
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int d = threadIdx.x; d < NBUK; d += RT)
    for (int w = 0; w < RT / 64; w++) cnt[w][d] = 0;
  __syncthreads();
  const i64 seg = (i64)blockIdx.x * (RT * RCH) + (i64)wv * (RCH * 64);
  uint32_t key[RCH], rank[RCH];
  int32_t val[RCH];
  rank_chunks<RCH>(kin, vin, n, shift, seg, lane, cnt[wv], key, val, rank);
  __syncthreads();
  for (int d = threadIdx.x; d < NBUK; d += RT) {
    uint32_t run = start[(i64)blockIdx.x * NBUK + d];
#pragma unroll
    for (int w = 0; w < RT / 64; w++) {
      uint32_t t = cnt[w][d];
      cnt[w][d] = run;
      run += t;
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < RCH; c++) {
    i64 i = seg + c * 64 + lane;
    if (i < n) {
      uint32_t d = (key[c] >> shift) & (NBUK - 1);
      uint32_t pos = cnt[wv][d] + rank[c];
      if (kout) kout[pos] = key[c];  // the last pass writes only the values
      vout[pos] = val[c];
    }
  }
}

// Per-pass tile starts in one launch: workgroup b owns digits 16 b .. +16, and its thread (tile group g of 64, digit)
// a run of consecutive tiles. Column sums give each digit's total, which is published (flag in the high word of a zeroed
// 64-bit slot); the digit's start is the sum of the lower digits' published totals, read back all at once (workgroups
// start in id order, so every lower digit's workgroup is already running and publishes without waiting). The wait is
// bounded: a total not published within spin_limit polls is summed by the waiting lane from the tile counts, so the
// result never depends on the schedule (the limit only trades waiting against re-reading). The columns then become
// exclusive tile starts in `start` (not in place: the counts stay intact for such a fallback read).
// It is bound by its dependent round trips, not by bytes. With digit-major counts and one workgroup per digit, every
// tile's 512 counts and starts were 512 separate lines, for the count and the scatter kernel too: 1.2 M keys, count
// 10.3 -> 6.6 us, scan 10.8 -> 9.2, scatter 10.8 -> 9.2. The held counts' loops end at the run's length, the same for all
// threads: walked to their full 32, builds of 25 to 60 k rows were 1 to 2 us slower than digit-major (40000 rows, whole
// build: digit-major 58.7, full walk 59.6, as it is 55.5).
constexpr int DPW = 16, TG = 64, HELD = 32;  // digits per workgroup, tile groups, counts held by a thread
__global__ void __launch_bounds__(DPW* TG) k_rs_digit_scan(const uint32_t* __restrict__ cnt,
                                                           uint32_t* __restrict__ start, uint64_t* __restrict__ dsum,
                                                           int ntiles, uint32_t spin_limit,
                                                           const uint32_t* __restrict__ ndev, int tile_keys) {
  __shared__ uint32_t part[DPW][TG + 1], tot[DPW], low[DPW];
  const int d0 = blockIdx.x * DPW, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (ndev) ntiles = max(1, min(ntiles, (int)(((i64)*ndev + tile_keys - 1) / tile_keys)));  // tiles with keys
  const int dd = tid % DPW, g = tid / DPW, per = (ntiles + TG - 1) / TG;
  const int t0 = min(g * per, ntiles), t1 = min(t0 + per, ntiles);
  const uint32_t* col = cnt + d0 + dd;
  uint32_t mine = 0, c[HELD] = {};  // a short run is read once, all of it in flight, and held; a long one read twice
  const bool held = per <= HELD;
  if (held) {
#pragma unroll
    for (int k0 = 0; k0 < HELD; k0 += 4) {
      if (k0 >= per) break;
#pragma unroll
      for (int k = k0; k < k0 + 4; k++) c[k] = t0 + k < t1 ? col[(i64)(t0 + k) * NBUK] : 0u;
    }
#pragma unroll
    for (int k = 0; k < HELD; k++) mine += c[k];
  } else {
#pragma unroll 8
    for (int t = t0; t < t1; t++) mine += col[(i64)t * NBUK];
  }
  part[dd][g] = mine;
  __syncthreads();
  static_assert(DPW == 16 && TG == 64 && NBUK <= DPW * TG, "one wavefront per digit, one published sum per thread");
  // wavefront wv: digit d0 + wv, lane = tile group
  const uint32_t v = part[wv][lane];
  uint32_t inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = (uint32_t)__shfl_up((int)inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) {
    __hip_atomic_store(dsum + d0 + wv, ST_SUM | inc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    tot[wv] = inc;
  }
  uint32_t below = 0;
  if (tid < d0) {  // the digits of the lower workgroups, one per thread
    uint64_t w = __hip_atomic_load(dsum + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (uint32_t spins = 0; (w >> 32) == 0 && spins < spin_limit; spins++)
      w = __hip_atomic_load(dsum + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((w >> 32) == 0) {
      // not published within the limit: sum the digit's tile counts here (they are complete: the count kernel ran
      // before this launch), so the start is exact whatever the workgroup schedule
      uint32_t s = 0;
      for (int t = 0; t < ntiles; t++) s += cnt[(i64)t * NBUK + tid];
      w = s;
    }
    below = (uint32_t)w;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) below += (uint32_t)__shfl_xor((int)below, o, 64);
  if (lane == 0) low[wv] = below;
  __syncthreads();
  uint32_t first = 0;
#pragma unroll
  for (int w = 0; w < DPW; w++) first += low[w] + (w < wv ? tot[w] : 0u);
  part[wv][lane] = first + inc - v;
  __syncthreads();
  uint32_t run = part[dd][g];
  uint32_t* out = start + d0 + dd;
  if (held) {
#pragma unroll
    for (int k0 = 0; k0 < HELD; k0 += 4) {
      if (k0 >= per) break;
#pragma unroll
      for (int k = k0; k < k0 + 4; k++) {
        if (t0 + k < t1) out[(i64)(t0 + k) * NBUK] = run;
        run += c[k];
      }
    }
    return;
  }
#pragma unroll 8
  for (int t = t0; t < t1; t++) {
    const uint32_t v = col[(i64)t * NBUK];
    out[(i64)t * NBUK] = run;
    run += v;
  }
}

// One pass in one launch, for few keys: every workgroup (1024 keys, one chunk per wavefront) counts the digits of all
// n keys itself, those of the tiles before its own apart, which gives its tile starts without a count and a scan
// launch; ranks and destinations are the scatter kernel's. The counting bounds it, and in it the lanes of a wavefront
// that add to one LDS counter: one after the other, up to 64 of them, since solid shapes hold mostly one mask and shells
// few. So the two digits held by the first lanes are each added once by one of their lanes (kernel map of 24000 rows:
// shell 58.5 -> 51.9 us, solid cube 84.9 -> 40.8, all children of 3000 parents 89.7 -> 66.5; one such digit 53.0 /
// 44.9 / 71.6, three 52.4 / 41.1 / 70).
__global__ void __launch_bounds__(1024) k_rs_pass(const uint32_t* __restrict__ kin, const int32_t* __restrict__ vin,
                                                  uint32_t* __restrict__ kout, int32_t* __restrict__ vout, int n,
                                                  int shift, const uint32_t* __restrict__ ndev) {
  constexpr int NW = 16, U = 4, LEAD = 2;
  __shared__ uint32_t cnt[NW][NBUK], before[NBUK], rest[NBUK], red[NBUK / 64];
  if (ndev) n = min((uint32_t)n, *ndev);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, base = blockIdx.x * 1024;
  if (base >= n) return;
  for (int d = lane; d < NBUK; d += 64) cnt[wv][d] = 0;
  if (tid < NBUK) before[tid] = rest[tid] = 0;
  __syncthreads();
  for (int i0 = 0; i0 < n; i0 += 1024 * U) {
    uint32_t k[U];
#pragma unroll
    for (int u = 0; u < U; u++) k[u] = i0 + u * 1024 + tid < n ? kin[i0 + u * 1024 + tid] : 0u;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i1 = i0 + u * 1024;
      if (i1 + tid >= n) break;
      uint32_t* c = i1 < base ? before : rest;
      const uint32_t d = (k[u] >> shift) & (NBUK - 1);
      bool mine = true;  // not added yet
#pragma unroll
      for (int l = 0; l < LEAD; l++) {
        if (!mine) break;
        const uint32_t first = __builtin_amdgcn_readfirstlane(d);
        const uint64_t peers = __ballot(d == first);
        if (d == first) {
          mine = false;
          if (lane == __builtin_ctzll(peers)) atomicAdd(&c[d], (uint32_t)__popcll(peers));
        }
      }
      if (mine) atomicAdd(&c[d], 1u);
    }
  }
  uint32_t key[1], rank[1];
  int32_t val[1];
  rank_chunks<1>(kin, vin, n, shift, base + wv * 64, lane, cnt[wv], key, val, rank);
  __syncthreads();
  uint32_t tot = 0, inc = 0;
  if (tid < NBUK) {
    inc = tot = before[tid] + rest[tid];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t t = (uint32_t)__shfl_up((int)inc, o, 64);
      if (lane >= o) inc += t;
    }
    if (lane == 63) red[wv] = inc;
  }
  __syncthreads();
  if (tid < NBUK) {
    uint32_t run = inc - tot + before[tid];
#pragma unroll
    for (int w = 0; w < NBUK / 64; w++) run += w < wv ? red[w] : 0u;
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const uint32_t t = cnt[w][tid];
      cnt[w][tid] = run;
      run += t;
    }
  }
  __syncthreads();
  if (base + tid < n) {
    const uint32_t pos = cnt[wv][(key[0] >> shift) & (NBUK - 1)] + rank[0];
    if (kout) kout[pos] = key[0];  // the last pass writes only the values
    vout[pos] = val[0];
  }
}
// Kernel map of n voxels, one launch per pass / three, us: shell 8000 36 / 53, 16000 44 / 54, 20000 47 / 54, 24000
// 52 / 53, 28000 56 / 55, 34000 62 / 55; all children kept 16000 60 / 73, 24000 67 / 75, 34000 78 / 77: counting all keys
// in every workgroup pays up to ~24 k of them.
constexpr i64 kSmallKeys = 1024 * 24;
}  // namespace

SortWork sort_work(i64 n, int bits, i64 likely) {
  SortWork w;
  w.passes = (bits + RBITS - 1) / RBITS;
  if (n <= kSmallKeys) return w;  // each pass counts for itself: no workspace, nothing to count
  // the largest tile that still leaves ~900 tiles (interleaved builds, one box: C3 0.390 M keys best at 4, C4 3.76 M
  // at 16 (8: +3%), C5's children 2.15 M at 8 (16: +1.2%))
  w.rch = likely >= (i64)RT * 16 * 900 ? 16 : (likely >= (i64)RT * 8 * 900 ? 8 : 4);
  w.ntiles = (int)std::max<i64>(cdiv(n, (i64)RT * w.rch), 1);
  w.zwords = (i64)w.passes * NBUK * 2 + (i64)NBUK * w.ntiles;
  // [digit-sum slots: passes x NBUK u64][first pass's counts: ntiles x NBUK][tile starts: ntiles x NBUK]; the
  // slot words are even in number, so the 64-bit slots and everything after them stay 8-byte aligned
  w.buf = empty({w.zwords + (i64)NBUK * w.ntiles}, I32);
  return w;
}

void stable_sort_pairs(const uint32_t* keys, const int32_t* vals, i64 n, int bits, int32_t* vals_out,
                       const uint32_t* ndev, SortWork* pre) {
  if (n <= 0) return;
  REQ(n < (1ll << 31), "sort size %lld", (long long)n);
  REQ(bits >= 1 && bits <= 32, "key bits %d", bits);
  hipStream_t s = stream();
  // SPCONV_SORT_SPIN_LIMIT overrides the digit-sum wait bound (0: every workgroup recomputes the lower digits' sums
  // itself; the tests use it to check that path)
  uint32_t spin_limit = kSpinLimit;
  if (const char* e = getenv("SPCONV_SORT_SPIN_LIMIT")) spin_limit = (uint32_t)strtoul(e, nullptr, 10);
  const bool small = n <= kSmallKeys;
  SortWork own;
  if (!pre) own = sort_work(n, bits, n);
  SortWork& w = pre ? *pre : own;
  REQ(w.passes == (bits + RBITS - 1) / RBITS &&
          (small ? w.rch == 0 : w.ntiles == (int)std::max<i64>(cdiv(n, (i64)RT * w.rch), 1)),
      "sort workspace made for another size");
  const int passes = w.passes, rch = w.rch, ntiles = w.ntiles;
  Tensor kb0 = empty({n}, I32), kb1 = empty({n}, I32), vb0 = empty({n}, I32), vb1 = empty({n}, I32);
  // ping-pong buffers; the last pass writes only its values, straight into vals_out
  const uint32_t* kin = keys;
  const int32_t* vin = vals;
  auto outs = [&](int p, uint32_t*& kout, int32_t*& vout) {
    kout = p + 1 == passes ? nullptr : ((p & 1) ? kb1.ptr<uint32_t>() : kb0.ptr<uint32_t>());
    vout = p + 1 == passes ? vals_out : ((p & 1) ? vb1.ptr<int32_t>() : vb0.ptr<int32_t>());
  };
  if (small) {
    for (int p = 0; p < passes; p++) {
      uint32_t* kout;
      int32_t* vout;
      outs(p, kout, vout);
      k_rs_pass<<<cdiv(n, 1024), 1024, 0, s>>>(kin, vin, kout, vout, (int)n, p * RBITS, ndev);
      kin = kout;
      vin = vout;
    }
    CK(hipGetLastError());
    return;
  }
  const i64 swords = (i64)passes * NBUK * 2;
  uint64_t* dsum = (uint64_t*)w.buf.ptr<uint32_t>();
  uint32_t* h = w.buf.ptr<uint32_t>() + swords;
  uint32_t* st = h + (i64)NBUK * ntiles;
  for (int p = 0; p < passes; p++) {
    uint32_t* kout;
    int32_t* vout;
    outs(p, kout, vout);
    const int shift = p * RBITS;
    if (p > 0 || !pre) {  // a caller-made workspace arrives with the first pass counted and the slots zeroed
      uint32_t* z = p == 0 ? (uint32_t*)dsum : nullptr;  // the first count kernel zeroes every pass's digit sums
      const int zn = (int)swords;
      if (rch == 16) k_rs_count<16><<<ntiles, RT, 0, s>>>(kin, n, shift, h, z, zn, ndev);
      else if (rch == 8) k_rs_count<8><<<ntiles, RT, 0, s>>>(kin, n, shift, h, z, zn, ndev);
      else k_rs_count<4><<<ntiles, RT, 0, s>>>(kin, n, shift, h, z, zn, ndev);
    }
    k_rs_digit_scan<<<NBUK / DPW, DPW * TG, 0, s>>>(h, st, dsum + p * NBUK, ntiles, spin_limit, ndev, RT * rch);
    if (rch == 16) k_rs_scatter<16><<<ntiles, RT, 0, s>>>(kin, vin, kout, vout, n, shift, st, ndev);
    else if (rch == 8) k_rs_scatter<8><<<ntiles, RT, 0, s>>>(kin, vin, kout, vout, n, shift, st, ndev);
    else k_rs_scatter<4><<<ntiles, RT, 0, s>>>(kin, vin, kout, vout, n, shift, st, ndev);
    kin = kout;
    vin = vout;
  }
  CK(hipGetLastError());
}

void stable_argsort27(const uint32_t* keys, i64 n, int32_t* order, const uint32_t* ndev, SortWork* pre) {
  stable_sort_pairs(keys, nullptr, n, 27, order, ndev, pre);
}
