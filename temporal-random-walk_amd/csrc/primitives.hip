// primitives.hip -- device-wide scan, stable LSD radix sort and reductions.
// See primitives.h for the design notes.
#include "primitives.h"

#include <algorithm>
#include <type_traits>

#include <stdexcept>
#include <string>

namespace trw {

void check_hip(hipError_t e, const char* what) {
    if (e != hipSuccess) {
        throw std::runtime_error(std::string("HIP error in ") + what + ": " +
                                 hipGetErrorString(e));
    }
}

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;

// Scan operators: a sum, and a running maximum (identity -inf).
struct OpSum {
    template <typename T>
    __device__ static T identity() { return T(0); }
    template <typename T>
    __device__ static T apply(T a, T b) { return a + b; }
};
struct OpMax {
    template <typename T>
    __device__ static T identity() { return -__builtin_huge_val(); }
    template <typename T>
    __device__ static T apply(T a, T b) { return a > b ? a : b; }
};

// ---------------------------------------------------------------------------
// block-level helpers (256 threads = 4 wave64, unless W says otherwise)
// ---------------------------------------------------------------------------
template <typename T, typename Op = OpSum>
__device__ __forceinline__ T wave_inclusive_scan(T x, int lane) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const T y = __shfl_up(x, off, 64);
        if (lane >= off) x = Op::apply(x, y);
    }
    return x;
}

// Exclusive block scan of one value per thread; *total receives the block
// total.  The exclusive value is built from the wave prefix and the shifted
// inclusive scan, so it is exact for the maximum as well as for integers.
template <typename T, typename Op = OpSum, int W = kWaves>
__device__ __forceinline__ T block_exclusive_scan(T v, T* total, T* s_wave) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const T inc = wave_inclusive_scan<T, Op>(v, lane);
    const T below = __shfl_up(inc, 1, 64);
    if (lane == 63) s_wave[wave] = inc;
    __syncthreads();
    T wp = Op::template identity<T>(), tot = Op::template identity<T>();
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const T sw = s_wave[w];
        if (w < wave) wp = Op::apply(wp, sw);
        tot = Op::apply(tot, sw);
    }
    __syncthreads();
    *total = tot;
    return lane == 0 ? wp : Op::apply(wp, below);
}

template <typename T, typename Op = OpSum>
__device__ __forceinline__ T block_sum(T v, T* s_wave) {
    T tot;
    (void)block_exclusive_scan<T, Op>(v, &tot, s_wave);
    return tot;
}

// ---------------------------------------------------------------------------
// scan: tile = 256 threads x 16 consecutive items per thread
//
// A thread owns 16 consecutive items, so that sums are rounded in one order
// whatever the launch; read that way a wave's access touches 64 lines of 128
// bytes for 512 bytes of doubles.  The tile therefore passes through LDS: memory
// is read and written in rows of 256 consecutive items, a thread's run is padded
// by one item (17 doubles apart, lanes hit distinct banks).  Same sums, bit for
// bit; bound by HBM.
// ---------------------------------------------------------------------------
constexpr int kScanItems = 16;
constexpr size_t kScanTile = static_cast<size_t>(kBlock) * kScanItems;
constexpr size_t kScanLds = kScanTile + kBlock;

// This thread's items of the tile at t0 (pad past n), through lds (kScanLds).
template <typename T>
__device__ __forceinline__ void scan_tile_load(const T* in, size_t t0, size_t n, T pad, T* lds,
                                               T (&v)[kScanItems]) {
#pragma unroll
    for (int r = 0; r < kScanItems; ++r) {
        const uint32_t i = r * kBlock + threadIdx.x;
        lds[i + i / kScanItems] = t0 + i < n ? in[t0 + i] : pad;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) v[j] = lds[threadIdx.x * (kScanItems + 1) + j];
}

// Writes the tile at t0 from the threads' items; lds was last read by
// scan_tile_load (a thread overwrites only what it has read itself).
template <typename T>
__device__ __forceinline__ void scan_tile_store(T* out, size_t t0, size_t n, T* lds,
                                                const T (&v)[kScanItems]) {
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) lds[threadIdx.x * (kScanItems + 1) + j] = v[j];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kScanItems; ++r) {
        const uint32_t i = r * kBlock + threadIdx.x;
        if (t0 + i < n) out[t0 + i] = lds[i + i / kScanItems];
    }
}

template <typename T, typename Op>
__global__ __launch_bounds__(kBlock) void scan_reduce_kernel(const T* __restrict__ in, size_t n,
                                                             T* __restrict__ sums) {
    __shared__ T s_wave[kWaves];
    __shared__ T s_tile[kScanLds];
    T v[kScanItems];
    scan_tile_load(in, blockIdx.x * kScanTile, n, Op::template identity<T>(), s_tile, v);
    T acc = Op::template identity<T>();
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) acc = Op::apply(acc, v[j]);
    const T tot = block_sum<T, Op>(acc, s_wave);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// Single block: exclusive scan of sums[0..nb) in place; sums[nb] = total.
template <typename T, typename Op>
__global__ __launch_bounds__(kBlock) void scan_sums_kernel(T* __restrict__ sums, size_t nb) {
    __shared__ T s_wave[kWaves];
    T carry = Op::template identity<T>();
    for (size_t chunk = 0; chunk < nb; chunk += kScanTile) {
        const size_t base = chunk + static_cast<size_t>(threadIdx.x) * kScanItems;
        T v[kScanItems];
        T acc = Op::template identity<T>();
#pragma unroll
        for (int j = 0; j < kScanItems; ++j) {
            const size_t i = base + j;
            v[j] = i < nb ? sums[i] : Op::template identity<T>();
            acc = Op::apply(acc, v[j]);
        }
        T tot;
        T run = Op::apply(carry, block_exclusive_scan<T, Op>(acc, &tot, s_wave));
#pragma unroll
        for (int j = 0; j < kScanItems; ++j) {
            const size_t i = base + j;
            if (i < nb) sums[i] = run;
            run = Op::apply(run, v[j]);
        }
        carry = Op::apply(carry, tot);
        __syncthreads();
    }
    if (threadIdx.x == 0) sums[nb] = carry;
}

template <typename T, bool Inclusive, typename Op>
__global__ __launch_bounds__(kBlock) void scan_apply_kernel(const T* in, T* out, size_t n,
                                                            const T* __restrict__ sums) {
    __shared__ T s_wave[kWaves];
    __shared__ T s_tile[kScanLds];
    const size_t t0 = blockIdx.x * kScanTile;
    T v[kScanItems];
    scan_tile_load(in, t0, n, Op::template identity<T>(), s_tile, v);
    T acc = Op::template identity<T>();
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) acc = Op::apply(acc, v[j]);
    T tot;
    T run = Op::apply(sums[blockIdx.x], block_exclusive_scan<T, Op>(acc, &tot, s_wave));
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        const T x = v[j];
        if (Inclusive) run = Op::apply(run, x);
        v[j] = run;
        if (!Inclusive) run = Op::apply(run, x);
    }
    scan_tile_store(out, t0, n, s_tile, v);
    if (!Inclusive && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = sums[gridDim.x];
}

// ---------------------------------------------------------------------------
// uint32 exclusive scan with coalesced accesses: the same 4096-item tiles, but
// wave w of a tile owns items [1024 w, 1024 w + 1024) as four rows of 256, and
// lane l holds items 4l..4l+3 of each row (one 16-byte access per lane and
// row, 1 KiB contiguous per wave access).  Integer sums are exact in any
// order, so the tile totals equal the blocked kernels'.
// ---------------------------------------------------------------------------
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ u32x4_t load_u32x4(const uint32_t* in, size_t i, size_t n) {
    if (i + 4 <= n) return *reinterpret_cast<const u32x4_t*>(in + i);
    u32x4_t v = {0u, 0u, 0u, 0u};
    if (i < n) v.x = in[i];
    if (i + 1 < n) v.y = in[i + 1];
    if (i + 2 < n) v.z = in[i + 2];
    return v;
}

__global__ __launch_bounds__(kBlock) void scan_reduce_u32_kernel(const uint32_t* __restrict__ in,
                                                                 size_t n,
                                                                 uint32_t* __restrict__ sums) {
    __shared__ uint32_t s_wave[kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t wbase = blockIdx.x * kScanTile + static_cast<size_t>(wave) * 1024 + lane * 4;
    uint32_t acc = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const u32x4_t v = load_u32x4(in, wbase + r * 256, n);
        acc += v.x + v.y + v.z + v.w;
    }
    const uint32_t tot = block_sum<uint32_t, OpSum>(acc, s_wave);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

__global__ __launch_bounds__(kBlock) void scan_apply_u32_kernel(const uint32_t* in,
                                                                uint32_t* out, size_t n,
                                                                const uint32_t* __restrict__ sums) {
    __shared__ uint32_t s_wave[kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t wbase = blockIdx.x * kScanTile + static_cast<size_t>(wave) * 1024 + lane * 4;
    u32x4_t v[4];
    uint32_t excl[4], row_tot[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = load_u32x4(in, wbase + r * 256, n);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint32_t ls = v[r].x + v[r].y + v[r].z + v[r].w;
        const uint32_t inc = wave_inclusive_scan<uint32_t, OpSum>(ls, lane);
        excl[r] = inc - ls;
        row_tot[r] = __shfl(inc, 63, 64);
    }
    const uint32_t wave_tot = row_tot[0] + row_tot[1] + row_tot[2] + row_tot[3];
    if (lane == 0) s_wave[wave] = wave_tot;
    __syncthreads();
    uint32_t carry = sums[blockIdx.x];
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
        if (w < wave) carry += s_wave[w];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const size_t i = wbase + r * 256;
        u32x4_t o;
        o.x = carry + excl[r];
        o.y = o.x + v[r].x;
        o.z = o.y + v[r].y;
        o.w = o.z + v[r].z;
        if (i + 4 <= n) {
            *reinterpret_cast<u32x4_t*>(out + i) = o;
        } else {
            if (i < n) out[i] = o.x;
            if (i + 1 < n) out[i + 1] = o.y;
            if (i + 2 < n) out[i + 2] = o.z;
        }
        carry += row_tot[r];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = sums[gridDim.x];
}

template <typename T, bool Inclusive, typename Op = OpSum>
void scan_impl(const T* in, T* out, size_t n, T* scratch, hipStream_t s) {
    if (n == 0) {
        if (!Inclusive) check_hip(hipMemsetAsync(out, 0, sizeof(T), s), "scan memset");
        return;
    }
    const size_t nb = (n + kScanTile - 1) / kScanTile;
    hipLaunchKernelGGL((scan_reduce_kernel<T, Op>), dim3(nb), dim3(kBlock), 0, s, in, n, scratch);
    hipLaunchKernelGGL((scan_sums_kernel<T, Op>), dim3(1), dim3(kBlock), 0, s, scratch, nb);
    hipLaunchKernelGGL((scan_apply_kernel<T, Inclusive, Op>), dim3(nb), dim3(kBlock), 0, s, in,
                       out, n, scratch);
    check_hip(hipGetLastError(), "scan launch");
}

// ---------------------------------------------------------------------------
// radix sort: a sort of B key bits splits them evenly over its passes (27 bits:
// four passes of 7).  The histogram kernel counts tiles of 4 waves x 8 rows x
// 64 keys = 2048 keys; a workgroup owns a few consecutive tiles, so the
// digit-major histogram has one column per workgroup (fewer scattered
// histogram writes and a shorter histogram scan per pass)
// ---------------------------------------------------------------------------
constexpr int kMaxDigitBits = 10;
constexpr int kRows = 8;
constexpr size_t kSortTile = static_cast<size_t>(kBlock) * kRows;
// The scatter's tile is 8 waves x 4 or 8 rows (sort_plan).
constexpr int kMaxTiles = 2;
constexpr int kScatterWaves = 8;
constexpr int kScatterBlock = kScatterWaves * 64;
constexpr int kRowsSmall = 4;
constexpr int kRowsLarge = 8;

__device__ __forceinline__ uint64_t lanes_below(int lane) {
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// Mask of the valid lanes of this wave whose digit (of db bits) equals mine.
__device__ __forceinline__ uint64_t match_digit(uint32_t d, bool valid, int db) {
    uint64_t m = __ballot(valid);
    for (int b = 0; b < db; ++b) {
        const bool bit = (d >> b) & 1u;
        const uint64_t vote = __ballot(bit);
        m &= bit ? vote : ~vote;
    }
    return m;
}

// A sort's input already in its buffers.
template <typename K, typename V>
struct PtrSource {
    const K* keys;
    const V* vals;  // may be null
    template <typename T>
    __device__ __forceinline__ T key_as(size_t i) const {
        return keys[i];
    }
    __device__ __forceinline__ V val(size_t i) const { return vals ? vals[i] : V(0); }
};

// Per-workgroup digit counts of keys[...] >> bit (db-bit digits, the digit
// masked to dmask), digit-major into hist.  Dynamic
// LDS: kWaves << db counters.
template <typename K, typename Src>
__global__ __launch_bounds__(kBlock) void radix_upsweep_kernel(Src in, size_t n, int bit, int db,
                                                               uint32_t dmask, int tiles,
                                                               uint32_t* __restrict__ hist,
                                                               size_t nb) {
    extern __shared__ uint32_t s_cnt[];  // [kWaves][R]
    const int R = 1 << db;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < kWaves * R; i += kBlock) s_cnt[i] = 0;
    __syncthreads();
    for (int t = 0; t < tiles; ++t) {
        const size_t wave_base = (static_cast<size_t>(blockIdx.x) * tiles + t) * kSortTile +
                                 static_cast<size_t>(wave) * kRows * 64;
        if (wave_base >= n) break;  // uniform over the wave
        K key[kRows];
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            const size_t i = wave_base + static_cast<size_t>(r) * 64 + lane;
            key[r] = i < n ? in.template key_as<K>(i) : K(0);
        }
        // counts only (no ranks): an LDS atomic per key, which a wave's
        // same-digit lanes serialise among themselves -- the row's lanes with
        // its first lane's digit add their count in one atomic (a hub's
        // node id fills half the rows of a power-law graph's node sort, and
        // their serialised atomics slowed that pass's histogram by 60 %)
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            const size_t i = wave_base + static_cast<size_t>(r) * 64 + lane;
            const uint32_t d = static_cast<uint32_t>(key[r] >> bit) & dmask;
            const bool valid = i < n;
            const uint64_t vm = __ballot(valid);
            if (vm == 0) continue;
            const int first = __ffsll(static_cast<long long>(vm)) - 1;
            const uint32_t d0 = __shfl(d, first, 64);
            const uint64_t m0 = __ballot(valid && d == d0);
            if (lane == first) atomicAdd(&s_cnt[wave * R + d0], static_cast<uint32_t>(__popcll(m0)));
            if (valid && d != d0) atomicAdd(&s_cnt[wave * R + d], 1u);
        }
    }
    __syncthreads();
    for (int d = threadIdx.x; d < R; d += kBlock) {
        uint32_t tot = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) tot += s_cnt[w * R + d];
        hist[static_cast<size_t>(d) * nb + blockIdx.x] = tot;
    }
}

// One workgroup per digit d: the exclusive scan of the workgroups' counts of
// digit d (hist[d * nb + b], in place), and the digit's total (the scatter adds
// the start of every digit, an exclusive scan of the totals).
__global__ __launch_bounds__(kBlock) void radix_offsets_kernel(uint32_t* __restrict__ hist,
                                                               size_t nb,
                                                               uint32_t* __restrict__ digit_tot) {
    __shared__ uint32_t s_wave[kWaves];
    uint32_t carry = 0;
    uint32_t* row = hist + static_cast<size_t>(blockIdx.x) * nb;
    for (size_t chunk = 0; chunk < nb; chunk += kScanTile) {
        const size_t base = chunk + static_cast<size_t>(threadIdx.x) * kScanItems;
        uint32_t v[kScanItems];
        uint32_t acc = 0;
#pragma unroll
        for (int j = 0; j < kScanItems; ++j) {
            const size_t i = base + j;
            v[j] = i < nb ? row[i] : 0u;
            acc += v[j];
        }
        uint32_t tot;
        uint32_t run = carry + block_exclusive_scan<uint32_t, OpSum>(acc, &tot, s_wave);
#pragma unroll
        for (int j = 0; j < kScanItems; ++j) {
            const size_t i = base + j;
            if (i < nb) row[i] = run;
            run += v[j];
        }
        carry += tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) digit_tot[blockIdx.x] = carry;
}

// The digit pass's LDS for a tile of W waves x Rows rows: W * R counters, R
// running positions, R output bases, then the tile's staged keys and values.
template <int W, int Rows, typename K, typename V>
struct TileLds {
    static constexpr size_t kTile = static_cast<size_t>(W) * Rows * 64;
    uint32_t* cnt;   // [W][R]: counts, then tile-local offsets
    uint32_t* run;   // the workgroup's next output position per digit
    uint32_t* base;  // output position of tile-local position 0, per digit
    K* key;
    V* val;
    __device__ __forceinline__ TileLds(uint32_t* lds, int R) {
        cnt = lds;
        run = cnt + W * R;
        base = run + R;
        key = reinterpret_cast<K*>(base + R);
        val = reinterpret_cast<V*>(key + kTile);
    }
    static constexpr size_t bytes(int R) {
        return (static_cast<size_t>(W) + 2) * R * sizeof(uint32_t) + kTile * (sizeof(K) + sizeof(V));
    }
};

// One tile's keys, values, digits and ranks in registers: row r of wave w is
// keys [(w * Rows + r) * 64, + 64) of the tile.
template <int Rows, typename K, typename V>
struct TileRegs {
    K key[Rows];
    V val[Rows];
    uint32_t dig[Rows];
    uint32_t rank[Rows];
};

template <int W, int Rows, typename K, typename V, typename Src>
__device__ __forceinline__ void tile_load(const Src& in, size_t n, size_t tile_base,
                                          TileRegs<Rows, K, V>& t) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t wave_base = tile_base + static_cast<size_t>(wave) * Rows * 64;
#pragma unroll
    for (int r = 0; r < Rows; ++r) {
        const size_t i = wave_base + static_cast<size_t>(r) * 64 + lane;
        const bool valid = i < n;
        t.key[r] = valid ? in.template key_as<K>(i) : K(0);
        t.val[r] = valid ? in.val(i) : V(0);
    }
}

// Ranks the loaded tile's keys by digit: rank = the number of earlier keys of
// the wave with the same digit; l.cnt[wave][d] ends as the wave's count of
// digit d.  The counters must be zero.
template <int W, int Rows, typename K, typename V>
__device__ __forceinline__ void tile_rank(size_t n, size_t tile_base, int bit, int db,
                                          uint32_t dmask, const TileLds<W, Rows, K, V>& l,
                                          TileRegs<Rows, K, V>& t) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, R = 1 << db;
    const size_t wave_base = tile_base + static_cast<size_t>(wave) * Rows * 64;
#pragma unroll
    for (int r = 0; r < Rows; ++r) {
        const size_t i = wave_base + static_cast<size_t>(r) * 64 + lane;
        const bool valid = i < n;
        const uint32_t d = static_cast<uint32_t>(t.key[r] >> bit) & dmask;
        t.dig[r] = d;
        const uint64_t m = match_digit(d, valid, db);
        const uint32_t before = __popcll(m & lanes_below(lane));
        const uint32_t prior = l.cnt[wave * R + d];
        t.rank[r] = prior + before;
        if (valid && before == 0) l.cnt[wave * R + d] = prior + __popcll(m);
    }
}

// Stages the ranked tile in LDS in its sorted order, l.cnt holding the
// tile-local start of every (wave, digit).
template <int W, int Rows, typename K, typename V>
__device__ __forceinline__ void tile_stage(size_t n, size_t tile_base, int db, bool with_vals,
                                           const TileLds<W, Rows, K, V>& l,
                                           const TileRegs<Rows, K, V>& t) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, R = 1 << db;
    const size_t wave_base = tile_base + static_cast<size_t>(wave) * Rows * 64;
#pragma unroll
    for (int r = 0; r < Rows; ++r) {
        const size_t i = wave_base + static_cast<size_t>(r) * 64 + lane;
        if (i < n) {
            const uint32_t lp = l.cnt[wave * R + t.dig[r]] + t.rank[r];
            l.key[lp] = t.key[r];
            if (with_vals) l.val[lp] = t.val[r];
        }
    }
}

// Writes the staged tile out by consecutive threads, so each digit's keys
// leave as one contiguous run: key lp goes to l.base[digit] + lp.  Store: the
// store (st) is written instead of keys_out / vals_out.
template <bool Store, int W, int Rows, typename K, typename V>
__device__ __forceinline__ void tile_write(size_t n, size_t tile_base, int bit, uint32_t dmask,
                                           const TileLds<W, Rows, K, V>& l, K* __restrict__ keys_out,
                                           V* __restrict__ vals_out, const SortedStore& st) {
    constexpr size_t kTile = TileLds<W, Rows, K, V>::kTile;
    const size_t tile_n = n - tile_base < kTile ? n - tile_base : kTile;
#pragma unroll
    for (int r = 0; r < Rows; ++r) {
        const uint32_t lp = static_cast<uint32_t>(r) * W * 64 + threadIdx.x;
        if (lp < tile_n) {
            const K k = l.key[lp];
            const uint32_t d = static_cast<uint32_t>(k >> bit) & dmask;
            const uint32_t pos = l.base[d] + lp;
            if constexpr (Store) {
                const uint64_t v = l.val[lp];
                st.src[pos] = static_cast<int32_t>(static_cast<uint32_t>(v));
                st.dst[pos] = static_cast<int32_t>(static_cast<uint32_t>(v >> 32));
                st.ts[pos] = static_cast<int64_t>(static_cast<uint64_t>(k) +
                                                  static_cast<uint64_t>(st.tmin));
            } else {
                keys_out[pos] = k;
                if (vals_out) vals_out[pos] = l.val[lp];
            }
        }
    }
}

// Stable scatter of one digit pass, `tiles` tiles per workgroup.  Dynamic LDS:
// TileLds::bytes.
template <typename K, typename V, int Rows, bool Store, typename Src>
__global__ __launch_bounds__(kScatterBlock) void radix_scatter_kernel(
    Src in, K* __restrict__ keys_out, V* __restrict__ vals_out, size_t n, int bit, int db, uint32_t dmask, int tiles,
    const uint32_t* __restrict__ offsets, size_t nb, const uint32_t* __restrict__ digit_tot,
    SortedStore st = SortedStore{}) {
    extern __shared__ __align__(16) uint32_t s_lds[];
    __shared__ uint32_t s_wave[kScatterWaves];
    const int R = 1 << db;
    constexpr size_t kTile = static_cast<size_t>(kScatterBlock) * Rows;
    const TileLds<kScatterWaves, Rows, K, V> l(s_lds, R);
    // digits [d0, d0 + per) of this thread in the tile epilogue
    const int per = (R + kScatterBlock - 1) / kScatterBlock;
    const int d0 = threadIdx.x * per;
    {
        // the workgroup's first output position of every digit: the keys of
        // smaller digits, then those of earlier workgroups
        uint32_t mine = 0;
        for (int j = 0; j < per; ++j)
            if (d0 + j < R) mine += digit_tot[d0 + j];
        uint32_t tot;
        uint32_t at = block_exclusive_scan<uint32_t, OpSum, kScatterWaves>(mine, &tot, s_wave);
        for (int j = 0; j < per; ++j) {
            const int d = d0 + j;
            if (d < R) {
                l.run[d] = at + offsets[static_cast<size_t>(d) * nb + blockIdx.x];
                at += digit_tot[d];
            }
        }
    }
    for (int t = 0; t < tiles; ++t) {
        const size_t tile_base = (static_cast<size_t>(blockIdx.x) * tiles + t) * kTile;
        if (tile_base >= n) break;  // uniform over the workgroup
        for (int i = threadIdx.x; i < kScatterWaves * R; i += kScatterBlock) l.cnt[i] = 0;
        __syncthreads();
        TileRegs<Rows, K, V> regs;
        tile_load<kScatterWaves>(in, n, tile_base, regs);
        tile_rank(n, tile_base, bit, db, dmask, l, regs);
        __syncthreads();
        {
            // tile epilogue: the tile-local start of every digit (an exclusive
            // scan of the tile's digit counts), its waves' offsets after it,
            // and the output position of local position 0 for the digit
            uint32_t cnt_mine = 0;
            for (int j = 0; j < per; ++j) {
                const int d = d0 + j;
                if (d < R) {
#pragma unroll
                    for (int w = 0; w < kScatterWaves; ++w) cnt_mine += l.cnt[w * R + d];
                }
            }
            uint32_t tot;
            uint32_t start = block_exclusive_scan<uint32_t, OpSum, kScatterWaves>(cnt_mine, &tot, s_wave);
            for (int j = 0; j < per; ++j) {
                const int d = d0 + j;
                if (d < R) {
                    const uint32_t first = start;
#pragma unroll
                    for (int w = 0; w < kScatterWaves; ++w) {
                        const uint32_t c = l.cnt[w * R + d];
                        l.cnt[w * R + d] = start;
                        start += c;
                    }
                    l.base[d] = l.run[d] - first;  // wraps back in pos = base + local
                    l.run[d] += start - first;
                }
            }
        }
        __syncthreads();
        // the store pass writes no vals_out
        tile_stage(n, tile_base, db, vals_out || Store, l, regs);
        __syncthreads();
        tile_write<Store>(n, tile_base, bit, dmask, l, keys_out, vals_out, st);
        __syncthreads();  // the counters and the staging are reused by the next tile
    }
}

// ---------------------------------------------------------------------------
// sorts of one tile: every digit pass in one workgroup
// ---------------------------------------------------------------------------
// A sort this small is latency only (launches, and each pass's chain of LDS
// phases), so the tile is spread over 16 waves of 2 rows and a digit has at
// most 8 bits (a digit per thread between the passes).  320 keys by 32 bits:
// 14 us against 51 us as three kernels per pass.
constexpr int kTileBlock = 1024;
constexpr int kTileWaves = kTileBlock / 64;
constexpr int kTileRows = 2;
constexpr size_t kTileKeys = static_cast<size_t>(kTileBlock) * kTileRows;
constexpr int kTileDigitBits = 8;

// The keys go round through LDS.  keys_out / vals_out may be the source's arrays.
template <typename K, typename V, bool Store, typename Src>
__global__ __launch_bounds__(kTileBlock) void radix_tile_sort_kernel(
    Src in, bool with_vals, K* keys_out, V* vals_out, uint32_t n, int begin_bit, int end_bit, int db,
    SortedStore st = SortedStore{}) {
    extern __shared__ __align__(16) uint32_t s_lds[];
    __shared__ uint32_t s_wave[kTileWaves];
    const int R = 1 << db;
    const TileLds<kTileWaves, kTileRows, K, V> l(s_lds, R);
    TileRegs<kTileRows, K, V> regs;
    tile_load<kTileWaves>(in, n, 0, regs);
    for (int i = threadIdx.x; i < R; i += kTileBlock) l.base[i] = 0;
    const int d = threadIdx.x;
    for (int bit = begin_bit; bit < end_bit; bit += db) {
        const int w = end_bit - bit < db ? end_bit - bit : db;
        const uint32_t dmask = (1u << w) - 1u;
        if (bit != begin_bit) {
            // the keys as the last pass left them (every wave's reads precede
            // the next staging: the barriers below)
            tile_load<kTileWaves>(PtrSource<K, V>{l.key, with_vals ? l.val : nullptr}, n, 0, regs);
        }
        for (int i = threadIdx.x; i < kTileWaves * R; i += kTileBlock) l.cnt[i] = 0;
        __syncthreads();
        tile_rank(n, 0, bit, db, dmask, l, regs);
        __syncthreads();
        uint32_t c = 0;
        if (d < R) {
#pragma unroll
            for (int q = 0; q < kTileWaves; ++q) c += l.cnt[q * R + d];
        }
        uint32_t tot;
        uint32_t start = block_exclusive_scan<uint32_t, OpSum, kTileWaves>(c, &tot, s_wave);
        if (d < R) {
#pragma unroll
            for (int q = 0; q < kTileWaves; ++q) {
                const uint32_t x = l.cnt[q * R + d];
                l.cnt[q * R + d] = start;
                start += x;
            }
        }
        __syncthreads();
        tile_stage(n, 0, db, with_vals, l, regs);
        __syncthreads();
    }
    tile_write<Store>(n, 0, 0, 0u, l, keys_out, vals_out, st);  // base[0] = 0: key lp to lp
}

// How a sort of n keys by `bits` bits runs with `words` words of scratch: in
// one workgroup when they fit its tile, else three kernels per pass.  Measured
// (us; keys with 64-bit values, uniform):
//  - Digits: up to 10 bits while launches are the cost (100k keys by 20 bits:
//    43 in two passes, 47 in three), up to 8 past kWideMax, where a wide
//    digit's short runs write partial lines (1M: 81 in two passes of 10 bits,
//    60 in three of 7; 20M: 772 and 542).
//  - Tiles: one per workgroup until kSortBlocks workgroups (a workgroup's
//    tiles run one after the other: 100k keys by 32 bits, 64 with one, 90 with
//    two, 145 with four), then two.
//  - Rows: 2048-key tiles keep more workgroups resident (9M keys by 20 bits:
//    216 against 230); from kLargeMin keys on the output no longer stays in
//    cache, and 4096-key tiles write longer runs (20M: 480 against 528; 50M by
//    27 bits: 1716 against 1996).
constexpr size_t kWideMax = size_t{1} << 19;
constexpr size_t kLargeMin = size_t{3} << 22;
constexpr int kDigitBits = 8;
constexpr size_t kSortBlocks = 1024;
constexpr size_t kLdsBytes = size_t{160} << 10;  // of a CU, and the most a workgroup may take

struct SortPlan {
    bool one_tile, large;
    int passes, db;
    int tiles;     // tiles per workgroup
    size_t nb;     // workgroups of a pass
    size_t words;  // scratch: per-workgroup counts, then the digit totals
};

SortPlan sort_plan(size_t n, int bits, size_t words) {
    SortPlan p{};
    p.one_tile = n <= kTileKeys;
    p.large = n >= kLargeMin;
    const int most = p.one_tile ? kTileDigitBits : n <= kWideMax ? kMaxDigitBits : kDigitBits;
    p.passes = (bits + most - 1) / most;
    p.db = (bits + p.passes - 1) / p.passes;
    if (p.one_tile) return p;
    const size_t tile = static_cast<size_t>(kScatterBlock) * (p.large ? kRowsLarge : kRowsSmall);
    const size_t R = size_t{1} << p.db, all = (n + tile - 1) / tile;
    for (p.tiles = 1;; p.tiles *= 2) {
        p.nb = (all + p.tiles - 1) / p.tiles;
        p.words = p.nb * R + R;
        if (p.tiles >= kMaxTiles || (p.nb <= kSortBlocks && p.words <= words)) return p;
    }
}

// One digit pass from `in`: histogram, offsets, scatter (st: the store to write
// instead of ko / vo, or nullptr).
template <int Rows, typename K, typename V, typename Src>
void launch_pass(const SortPlan& p, const Src& in, K* ko, V* vo, size_t n, int bit, uint32_t dmask,
                 uint32_t* hist, const SortedStore* st, hipStream_t s) {
    const size_t R = size_t{1} << p.db;
    uint32_t* totals = hist + p.nb * R;
    const int up_tiles = static_cast<int>(p.tiles * (kScatterBlock * Rows / kSortTile));
    static_assert(kScatterBlock * kRowsSmall % kSortTile == 0, "whole histogram tiles");
    hipLaunchKernelGGL((radix_upsweep_kernel<K, Src>), dim3(p.nb), dim3(kBlock),
                       kWaves * R * sizeof(uint32_t), s, in, n, bit, p.db, dmask, up_tiles, hist,
                       p.nb);
    hipLaunchKernelGGL(radix_offsets_kernel, dim3(R), dim3(kBlock), 0, s, hist, p.nb, totals);
    using Lds = TileLds<kScatterWaves, Rows, K, V>;
    // 64-bit keys and values take 72 KiB at 10-bit digits, 74 KiB with large tiles
    // at 8: two such workgroups fit a CU
    static_assert(Lds::bytes(1 << (Rows == kRowsLarge ? kDigitBits : kMaxDigitBits)) <= kLdsBytes / 2,
                  "two workgroups per CU");
    const size_t lds = Lds::bytes(1 << p.db);
    if constexpr (std::is_same<V, uint64_t>::value) {
        if (st) {
            hipLaunchKernelGGL((radix_scatter_kernel<K, V, Rows, true, Src>), dim3(p.nb),
                               dim3(kScatterBlock), lds, s, in, nullptr, nullptr, n, bit, p.db, dmask,
                               p.tiles, hist, p.nb, totals, *st);
            return;
        }
    }
    hipLaunchKernelGGL((radix_scatter_kernel<K, V, Rows, false, Src>), dim3(p.nb),
                       dim3(kScatterBlock), lds, s, in, ko, vo, n, bit, p.db, dmask, p.tiles, hist,
                       p.nb, totals);
}

template <typename K, typename V, typename Src>
__global__ __launch_bounds__(kBlock) void source_copy_kernel(Src in, size_t n, K* __restrict__ keys,
                                                             V* __restrict__ vals) {
    const size_t i = blockIdx.x * static_cast<size_t>(kBlock) + threadIdx.x;
    if (i >= n) return;
    keys[i] = in.template key_as<K>(i);
    vals[i] = in.val(i);
}

// Sorts the n pairs of `in`, which is (keys0, vals0) itself for a PtrSource.
// Returns which buffer holds the result (-1: the store was written).
template <typename K, typename V, typename Src>
int radix_sort_impl(const Src& in, K* keys0, V* vals0, K* keys1, V* vals1, size_t n,
                    int begin_bit, int end_bit, RadixTmp tmp, hipStream_t s,
                    const SortedStore* store = nullptr) {
    constexpr bool in_place = std::is_same<Src, PtrSource<K, V>>::value;
    if (n <= 1 || end_bit <= begin_bit) {
        if (!in_place && n) {
            hipLaunchKernelGGL((source_copy_kernel<K, V, Src>), dim3((n + kBlock - 1) / kBlock),
                               dim3(kBlock), 0, s, in, n, keys0, vals0);
            check_hip(hipGetLastError(), "radix sort launch");
        }
        return 0;
    }
    const SortPlan p = sort_plan(n, end_bit - begin_bit, tmp.n);
    if (p.words > tmp.n) throw std::runtime_error("radix sort: scratch too small");
    K* kb[2] = {keys0, keys1};
    V* vb[2] = {vals0, vals1};
    const bool with_vals = !in_place || vals0 != nullptr;
    if (p.one_tile) {
        const size_t lds = TileLds<kTileWaves, kTileRows, K, V>::bytes(1 << p.db);
        const int out = p.passes & 1;
        bool stored = false;
        if constexpr (std::is_same<V, uint64_t>::value) {
            if (store) {
                hipLaunchKernelGGL((radix_tile_sort_kernel<K, V, true, Src>), dim3(1),
                                   dim3(kTileBlock), lds, s, in, with_vals, nullptr, nullptr,
                                   static_cast<uint32_t>(n), begin_bit, end_bit, p.db, *store);
                stored = true;
            }
        }
        if (!stored)
            hipLaunchKernelGGL((radix_tile_sort_kernel<K, V, false, Src>), dim3(1),
                               dim3(kTileBlock), lds, s, in, with_vals, kb[out], vb[out],
                               static_cast<uint32_t>(n), begin_bit, end_bit, p.db);
        check_hip(hipGetLastError(), "radix sort launch");
        return stored ? -1 : out;
    }
    int cur = 0;
    for (int pass = 0; pass < p.passes; ++pass) {
        const int bit = begin_bit + pass * p.db;
        // the last digit stops at end_bit
        const int w = end_bit - bit < p.db ? end_bit - bit : p.db;
        const uint32_t dmask = (1u << w) - 1u;
        const SortedStore* st = pass == p.passes - 1 ? store : nullptr;
        auto run = [&](const auto& from) {
            if (p.large)
                launch_pass<kRowsLarge>(p, from, kb[cur ^ 1], vb[cur ^ 1], n, bit, dmask, tmp.p, st, s);
            else
                launch_pass<kRowsSmall>(p, from, kb[cur ^ 1], vb[cur ^ 1], n, bit, dmask, tmp.p, st, s);
        };
        if (pass == 0) run(in);
        else run(PtrSource<K, V>{kb[cur], vb[cur]});
        check_hip(hipGetLastError(), "radix sort launch");
        cur ^= 1;
    }
    return store ? -1 : cur;
}

// ---------------------------------------------------------------------------
// group starts: exclusive scan of the spans' counts (one workgroup: 20M
// positions are 9766 spans)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void group_scan_kernel(uint32_t* __restrict__ v, size_t n,
                                                          uint32_t* __restrict__ total_out) {
    __shared__ uint32_t s_wave[16];
    uint32_t carry = 0;
    for (size_t c = 0; c < n; c += 4096) {
        const size_t i = c + threadIdx.x * 4u;
        const u32x4_t x = i < n ? load_u32x4(v, i, n) : u32x4_t{0u, 0u, 0u, 0u};
        uint32_t tot;
        uint32_t at = carry + block_exclusive_scan<uint32_t, OpSum, 16>(x.x + x.y + x.z + x.w, &tot,
                                                                        s_wave);
        const uint32_t y[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (i + k < n) v[i + k] = at;
            at += y[k];
        }
        carry += tot;
    }
    if (threadIdx.x == 0) *total_out = carry;
}

// ---------------------------------------------------------------------------
// reductions (grid-stride, per-block partials, then one block)
// ---------------------------------------------------------------------------
constexpr int kReduceBlocks = 1024;

// min and max of v, and the smallest of the ids a[i], b[i] (INT64_MAX for
// n == 0): one pass over a batch's timestamps and endpoints
struct MinMaxId {
    int64_t mn, mx, id, idmax;
};

__device__ __forceinline__ MinMaxId minmax_id_join(MinMaxId x, MinMaxId y) {
    return {y.mn < x.mn ? y.mn : x.mn, y.mx > x.mx ? y.mx : x.mx, y.id < x.id ? y.id : x.id,
            y.idmax > x.idmax ? y.idmax : x.idmax};
}

__device__ __forceinline__ MinMaxId block_minmax_id(MinMaxId v, int64_t* sm) {
    int64_t* m = sm + 4 * threadIdx.x;
    m[0] = v.mn;
    m[1] = v.mx;
    m[2] = v.id;
    m[3] = v.idmax;
    __syncthreads();
    for (int st = kBlock / 2; st > 0; st >>= 1) {
        if (static_cast<int>(threadIdx.x) < st) {
            const int64_t* o = sm + 4 * (threadIdx.x + st);
            const MinMaxId r = minmax_id_join({m[0], m[1], m[2], m[3]}, {o[0], o[1], o[2], o[3]});
            m[0] = r.mn;
            m[1] = r.mx;
            m[2] = r.id;
            m[3] = r.idmax;
        }
        __syncthreads();
    }
    return {sm[0], sm[1], sm[2], sm[3]};
}

__global__ __launch_bounds__(kBlock) void minmax_partial_kernel(const int64_t* __restrict__ v,
                                                                const int32_t* __restrict__ a,
                                                                const int32_t* __restrict__ b,
                                                                size_t n, int64_t* part) {
    __shared__ int64_t sm[4 * kBlock];
    MinMaxId acc{INT64_MAX, INT64_MIN, INT64_MAX, INT64_MIN};
    for (size_t i = blockIdx.x * static_cast<size_t>(kBlock) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * kBlock) {
        const int64_t x = v[i];
        const int32_t p = a[i], q = b[i];
        acc = minmax_id_join(acc, {x, x, min(p, q), max(p, q)});
    }
    const MinMaxId r = block_minmax_id(acc, sm);
    if (threadIdx.x == 0) {
        int64_t* o = part + 4 * blockIdx.x;
        o[0] = r.mn;
        o[1] = r.mx;
        o[2] = r.id;
        o[3] = r.idmax;
    }
}

__global__ __launch_bounds__(kBlock) void minmax_final_kernel(const int64_t* part, int np,
                                                              int64_t* out) {
    __shared__ int64_t sm[4 * kBlock];
    MinMaxId acc{INT64_MAX, INT64_MIN, INT64_MAX, INT64_MIN};
    for (int i = threadIdx.x; i < np; i += kBlock) {
        const int64_t* p = part + 4 * i;
        acc = minmax_id_join(acc, {p[0], p[1], p[2], p[3]});
    }
    const MinMaxId r = block_minmax_id(acc, sm);
    if (threadIdx.x == 0) {
        out[0] = r.mn;
        out[1] = r.mx;
        out[2] = r.id;
        out[3] = r.idmax;
    }
}

__global__ __launch_bounds__(kBlock) void max_pair_kernel(const int32_t* __restrict__ a,
                                                          const int32_t* __restrict__ b, size_t n,
                                                          int32_t* out) {
    __shared__ int32_t s[kBlock];
    int32_t mx = -1;
    for (size_t i = blockIdx.x * static_cast<size_t>(kBlock) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * kBlock) {
        mx = max(mx, max(a[i], b[i]));
    }
    s[threadIdx.x] = mx;
    __syncthreads();
    for (int st = kBlock / 2; st > 0; st >>= 1) {
        if (static_cast<int>(threadIdx.x) < st) s[threadIdx.x] = max(s[threadIdx.x], s[threadIdx.x + st]);
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicMax(out, s[0]);
}

__global__ void set_i32_kernel(int32_t* p, int32_t v) { *p = v; }

__global__ __launch_bounds__(kBlock) void sum_partial_kernel(const double* __restrict__ v,
                                                             size_t n, double* part) {
    __shared__ double s_wave[kWaves];
    double acc = 0.0;
    for (size_t i = blockIdx.x * static_cast<size_t>(kBlock) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * kBlock) {
        acc += v[i];
    }
    const double tot = block_sum(acc, s_wave);
    if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

__global__ __launch_bounds__(kBlock) void sum_final_kernel(const double* part, int np,
                                                           double* out) {
    __shared__ double s_wave[kWaves];
    double acc = 0.0;
    for (int i = threadIdx.x; i < np; i += kBlock) acc += part[i];
    const double tot = block_sum(acc, s_wave);
    if (threadIdx.x == 0) out[0] = tot;
}

int reduce_blocks(size_t n) {
    const size_t b = (n + kBlock - 1) / kBlock;
    return static_cast<int>(b < kReduceBlocks ? (b ? b : 1) : kReduceBlocks);
}

}  // namespace

size_t scan_scratch_elems(size_t n) { return (n + kScanTile - 1) / kScanTile + 1; }
// A sort's need does not grow with n throughout: it falls where digits become
// narrower (past kWideMax), where workgroups take two tiles (past kSortBlocks
// of them) and where tiles become larger (from kLargeMin on).  The scratch of n
// keys is therefore the largest of n's own and of the need just below each of
// those sizes.
static size_t scratch_words(size_t n, int bits, size_t words) {
    if (n <= 1 || bits <= 0) return 1;
    size_t most = 1;
    for (const size_t m : {n, kWideMax, kSortBlocks * kScatterBlock * kRowsSmall, kLargeMin - 1})
        if (m <= n) most = std::max(most, sort_plan(m, bits, words).words);
    return most;
}
size_t radix_tmp_elems(size_t n, int bits) { return scratch_words(n, bits, SIZE_MAX); }
size_t radix_min_elems(size_t n, int bits) { return scratch_words(n, bits, 0); }

void exclusive_scan_u32(const uint32_t* in, uint32_t* out, size_t n, uint32_t* scratch,
                        hipStream_t s) {
    // the coalesced kernels need 16-byte aligned arrays
    if (n == 0 || (reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) % 16) {
        scan_impl<uint32_t, false>(in, out, n, scratch, s);
        return;
    }
    const size_t nb = (n + kScanTile - 1) / kScanTile;
    hipLaunchKernelGGL(scan_reduce_u32_kernel, dim3(nb), dim3(kBlock), 0, s, in, n, scratch);
    hipLaunchKernelGGL((scan_sums_kernel<uint32_t, OpSum>), dim3(1), dim3(kBlock), 0, s, scratch,
                       nb);
    hipLaunchKernelGGL(scan_apply_u32_kernel, dim3(nb), dim3(kBlock), 0, s, in, out, n, scratch);
    check_hip(hipGetLastError(), "scan launch");
}
void exclusive_scan_u64(const uint64_t* in, uint64_t* out, size_t n, uint64_t* scratch,
                        hipStream_t s) {
    scan_impl<uint64_t, false>(in, out, n, scratch, s);
}
void inclusive_scan_f64(double* data, size_t n, double* scratch, hipStream_t s) {
    scan_impl<double, true>(data, data, n, scratch, s);
}
void running_max_f64(double* data, size_t n, double* scratch, hipStream_t s) {
    scan_impl<double, true, OpMax>(data, data, n, scratch, s);
}

int radix_sort_u64(uint64_t* keys0, uint32_t* vals0, uint64_t* keys1, uint32_t* vals1, size_t n,
                   int begin_bit, int end_bit, RadixTmp tmp, hipStream_t s) {
    return radix_sort_impl(PtrSource<uint64_t, uint32_t>{keys0, vals0}, keys0, vals0, keys1, vals1, n,
                           begin_bit, end_bit, tmp, s);
}
int radix_sort_u32(uint32_t* keys0, uint32_t* vals0, uint32_t* keys1, uint32_t* vals1, size_t n,
                   int begin_bit, int end_bit, RadixTmp tmp, hipStream_t s) {
    return radix_sort_impl(PtrSource<uint32_t, uint32_t>{keys0, vals0}, keys0, vals0, keys1, vals1, n,
                           begin_bit, end_bit, tmp, s);
}
int radix_sort_ts_u32(const TsSource& in, uint32_t* keys0, uint64_t* vals0, uint32_t* keys1,
                      uint64_t* vals1, size_t n, int bits, RadixTmp tmp, hipStream_t s,
                      const SortedStore* store) {
    return radix_sort_impl(in, keys0, vals0, keys1, vals1, n, 0, bits, tmp, s, store);
}
int radix_sort_ts_u64(const TsSource& in, uint64_t* keys0, uint64_t* vals0, uint64_t* keys1,
                      uint64_t* vals1, size_t n, int bits, RadixTmp tmp, hipStream_t s,
                      const SortedStore* store) {
    return radix_sort_impl(in, keys0, vals0, keys1, vals1, n, 0, bits, tmp, s, store);
}
int radix_sort_entries(const EntrySource& in, uint32_t* keys0, uint64_t* vals0, uint32_t* keys1,
                       uint64_t* vals1, size_t n, int bits, RadixTmp tmp, hipStream_t s) {
    auto sort = [&](const auto& from) {
        return radix_sort_impl(from, keys0, vals0, keys1, vals1, n, 0, bits, tmp, s);
    };
    if (in.mode == 0) return sort(EntrySourceOf<0>(in));
    if (in.mode == 1) return sort(EntrySourceOf<1>(in));
    return sort(EntrySourceOf<2>(in));
}
void group_scan(uint32_t* spans, size_t n_spans, uint32_t* host, hipStream_t s) {
    hipLaunchKernelGGL(group_scan_kernel, dim3(1), dim3(1024), 0, s, spans, n_spans, host);
    check_hip(hipGetLastError(), "group scan launch");
}
int radix_passes(size_t n, int begin_bit, int end_bit) {
    return n > 1 && end_bit > begin_bit ? sort_plan(n, end_bit - begin_bit, SIZE_MAX).passes : 0;
}
void minmax_ts_min_id(const int64_t* v, const int32_t* a, const int32_t* b, size_t n, int64_t* part,
                      int64_t* out, hipStream_t s) {
    const int nb = reduce_blocks(n);
    hipLaunchKernelGGL(minmax_partial_kernel, dim3(nb), dim3(kBlock), 0, s, v, a, b, n, part);
    hipLaunchKernelGGL(minmax_final_kernel, dim3(1), dim3(kBlock), 0, s, part, nb, out);
    check_hip(hipGetLastError(), "minmax launch");
}

void max_i32_pair(const int32_t* a, const int32_t* b, size_t n, int32_t* out, hipStream_t s) {
    hipLaunchKernelGGL(set_i32_kernel, dim3(1), dim3(1), 0, s, out, -1);
    if (n) {
        hipLaunchKernelGGL(max_pair_kernel, dim3(reduce_blocks(n)), dim3(kBlock), 0, s, a, b, n,
                           out);
    }
    check_hip(hipGetLastError(), "max launch");
}

// Scratch for the sum lives behind out (1024 doubles beyond out[0..1]).
void sum_f64(const double* v, size_t n, double* out, hipStream_t s) {
    const int nb = reduce_blocks(n);
    double* part = out + 2;
    hipLaunchKernelGGL(sum_partial_kernel, dim3(nb), dim3(kBlock), 0, s, v, n, part);
    hipLaunchKernelGGL(sum_final_kernel, dim3(1), dim3(kBlock), 0, s, part, nb, out);
    check_hip(hipGetLastError(), "sum launch");
}

}  // namespace trw
