// primitives.h -- device-wide scan and stable radix sort for the index build.
//
// Hand-written for CDNA4 (wave64): no rocPRIM / hipCUB.  The radix sort is a
// classic LSD sort with three launches per digit pass (tile histograms; one
// workgroup per digit scanning its histogram row; stable scatter), or one launch
// in all for inputs of one tile; a sort of B key bits takes the fewest passes
// of at most 8-bit digits (10-bit where launches outweigh the data), the bits
// split evenly.  Stable ranking inside a tile uses wave-level
// multisplit: one 64-lane ballot per digit bit gives every lane the mask of
// lanes holding the same digit, so the in-row rank is a popcount and a single
// leader lane per digit bumps the wave's LDS counter.  Waves own
// consecutive rows of the tile, so the scatter keeps input order among equal
// digits -- which is what makes the edge-store order "stable by (timestamp,
// insertion position)" and the node index "stable by (node, position)".
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace trw {

void check_hip(hipError_t e, const char* what);

// ---- scan ------------------------------------------------------------------
// Exclusive scan of n values given by an input functor; writes n + 1 outputs,
// out[n] = total.  `scratch` must hold scan_scratch_elems(n) elements of T.
size_t scan_scratch_elems(size_t n);

// Exclusive scan of a plain array: out[0..n] (out may alias in only if
// out != in is not required: in-place is supported).
void exclusive_scan_u32(const uint32_t* in, uint32_t* out, size_t n, uint32_t* scratch,
                        hipStream_t s);
void exclusive_scan_u64(const uint64_t* in, uint64_t* out, size_t n, uint64_t* scratch,
                        hipStream_t s);
// Inclusive scan of doubles in place (out[i] = in[0] + ... + in[i]).
void inclusive_scan_f64(double* data, size_t n, double* scratch, hipStream_t s);
// Running maximum of doubles in place (out[i] = max(in[0..i])): makes a
// cumulative array non-decreasing to the last ulp, whatever order its partial
// sums were rounded in.
void running_max_f64(double* data, size_t n, double* scratch, hipStream_t s);

// ---- radix sort --------------------------------------------------------------
// Stable sort of (key, value) pairs by key bits [begin_bit, end_bit).  Values
// may be null (keys only).  Buffers are ping-ponged; the function returns 0 if
// the sorted result ended in (keys0, vals0) and 1 if in (keys1, vals1).
// tmp: device scratch; radix_tmp_elems(n, end_bit - begin_bit) words let a sort
// of n keys, or of any fewer, run its fastest form, radix_min_elems words let it
// run.
struct RadixTmp {
    uint32_t* p;
    size_t n;  // words
};
size_t radix_tmp_elems(size_t n, int bits);
size_t radix_min_elems(size_t n, int bits);
int radix_sort_u64(uint64_t* keys0, uint32_t* vals0, uint64_t* keys1, uint32_t* vals1, size_t n,
                   int begin_bit, int end_bit, RadixTmp tmp, hipStream_t s);
int radix_sort_u32(uint32_t* keys0, uint32_t* vals0, uint32_t* keys1, uint32_t* vals1, size_t n,
                   int begin_bit, int end_bit, RadixTmp tmp, hipStream_t s);
// Digit passes of a sort of n keys by bits [begin_bit, end_bit) with
// radix_tmp_elems words of scratch: the result lands in buffer set (passes % 2).
int radix_passes(size_t n, int begin_bit, int end_bit);

// The edge store as the last pass of a sort of (timestamp key, packed
// endpoints) writes it: src = low half, dst = high half of the value, ts =
// key + tmin, each at the record's sorted position.
struct SortedStore {
    int32_t* src;
    int32_t* dst;
    int64_t* ts;
    int64_t tmin;
};
// Sources of a sort's input: its first digit pass reads the keys and values
// straight from the arrays they are made of, instead of from a copy a kernel
// would have to write (20M edges: 112 us for the timestamp keys, 79 us per
// direction for the entries).
//
// Edges keyed by timestamp: key ts - tmin, value the packed endpoints.
struct TsSource {
    const int64_t* ts;
    const int32_t* src;
    const int32_t* dst;
    int64_t tmin;
    template <typename K>
    __device__ __forceinline__ K key_as(size_t i) const {
        return static_cast<K>(static_cast<uint64_t>(ts[i]) - static_cast<uint64_t>(tmin));
    }
    __device__ __forceinline__ uint64_t val(size_t i) const {
        return static_cast<uint64_t>(static_cast<uint32_t>(src[i])) |
               (static_cast<uint64_t>(static_cast<uint32_t>(dst[i])) << 32);
    }
};
// Node-index entries of the edges src/dst, whose ids (store positions) start at
// id0: key = the list's node, value = the entry's walk record (neighbour in the
// low word, edge id in the high word: EdgeRec's layout), carried through the
// node sort so no record needs a gather afterwards.
// mode 0: out-lists (node = source, neighbour = target); 1: in-lists (node =
// target, neighbour = source); 2: undirected, entry 2i = (src_i; dst_i) and
// entry 2i+1 = (dst_i; src_i) (node_edge_index.cu:306-321) -- the neighbour is
// the reference's pick_other_number (utils/utils.cuh:102-104) seen from the
// entry's node.
// With erank given, a value packs the neighbour, the edge id and the edge's
// time key into one word (nbr | eid << nb | key << (nb + eb); the caller checks
// that they fit), so that the entries leave the node sort with their keys and
// the group flags need no gather of erank in node order.
struct EntrySource {
    const int32_t* src;
    const int32_t* dst;
    int mode;
    uint32_t id0;
    const uint32_t* erank;
    int nb, eb;
};
// The same for one mode.
template <int Mode>
struct EntrySourceOf : EntrySource {
    explicit EntrySourceOf(const EntrySource& e) : EntrySource(e) {}
    template <typename K>
    __device__ __forceinline__ K key_as(size_t i) const {
        const int32_t* p = Mode == 0 || (Mode == 2 && !(i & 1)) ? src : dst;
        return static_cast<K>(static_cast<uint32_t>(p[Mode == 2 ? i >> 1 : i]));
    }
    __device__ __forceinline__ uint64_t val(size_t i) const {
        const size_t e = Mode == 2 ? i >> 1 : i;
        const int32_t* p = Mode == 0 || (Mode == 2 && !(i & 1)) ? dst : src;
        const uint64_t nbr = static_cast<uint32_t>(p[e]);
        const uint64_t id = id0 + static_cast<uint32_t>(e);
        return erank ? nbr | (id << nb) | (static_cast<uint64_t>(erank[id]) << (nb + eb))
                     : nbr | (id << 32);
    }
};
// Sorts of a source's n pairs: as the sorts above with the source as (keys0,
// vals0), which are only written to.  store (may be null): the sort writes it
// instead; returns -1 then, unless it has no pass (n <= 1 or no key bits).
int radix_sort_ts_u32(const TsSource& in, uint32_t* keys0, uint64_t* vals0, uint32_t* keys1,
                      uint64_t* vals1, size_t n, int bits, RadixTmp tmp, hipStream_t s,
                      const SortedStore* store);
int radix_sort_ts_u64(const TsSource& in, uint64_t* keys0, uint64_t* vals0, uint64_t* keys1,
                      uint64_t* vals1, size_t n, int bits, RadixTmp tmp, hipStream_t s,
                      const SortedStore* store);
int radix_sort_entries(const EntrySource& in, uint32_t* keys0, uint64_t* vals0, uint32_t* keys1,
                       uint64_t* vals1, size_t n, int bits, RadixTmp tmp, hipStream_t s);

// ---- group starts ------------------------------------------------------------
// Groups of consecutive positions are marked by one bit per position (64 per
// word) and counted per kGroupSpan positions; position n's word always exists
// (its bit is 0).  group_scan turns the counts into the groups before each span
// (in place) and writes the total to host (pinned memory).
constexpr size_t kGroupSpan = 2048;
__host__ __device__ inline size_t group_words(size_t n) { return n / 64 + 1; }
__host__ __device__ inline size_t group_spans(size_t n) { return n / kGroupSpan + 1; }
void group_scan(uint32_t* spans, size_t n_spans, uint32_t* host, hipStream_t s);

// ---- reductions ---------------------------------------------------------------
// out[0], out[1] = min and max of v[0..n); out[2], out[3] = the smallest and
// the largest of a[i], b[i] (INT64_MAX / INT64_MIN when n == 0); out may be
// pinned host memory; part: minmax_scratch_elems() values of scratch
void minmax_ts_min_id(const int64_t* v, const int32_t* a, const int32_t* b, size_t n, int64_t* part,
                      int64_t* out, hipStream_t s);
inline size_t minmax_scratch_elems() { return 4 * 1024; }
// max of two int32 arrays -> *out (device memory); -1 when n == 0.
void max_i32_pair(const int32_t* a, const int32_t* b, size_t n, int32_t* out, hipStream_t s);
// sum of doubles -> *out (device memory).
void sum_f64(const double* v, size_t n, double* out, hipStream_t s);

}  // namespace trw
