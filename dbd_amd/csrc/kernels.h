// Host-side launchers for the gfx950 kernels in kernels.hip.
//
// Every row kernel is grid-stride over a "bin" (list of row ids), and reads the bin's
// [begin, end) from device memory (two int64 slots). The plain pipeline launches exactly as
// many workgroups as the bin needs; the batched/graph pipeline launches a fixed persistent
// grid that drains the same ranges, so nothing depends on host-side counts.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dbd {

constexpr int kMaxCats = 16;

// Category thresholds: row key k -> the number of limits below it, i.e. the smallest c with k <=
// lim[c] (c = 0 is "k == 0"). The limits of the last categories and of those past n are INT64_MAX.
struct CatTable {
  int64_t lim[kMaxCats];
  int32_t n;  // number of categories including 0 and the long category
};

struct Mat {
  const int64_t* ptr;
  const int32_t* idx;
  const void* val;
  int64_t nrows, ncols, nnz;
  // For A only: per-nonzero descriptor of the B row it selects (start, length), written by the
  // row analysis in A's order so later passes read it sequentially instead of gathering B.ptr.
  const int64_t* bstart = nullptr;
  const int32_t* blen = nullptr;
  // For B only: the band index of its long rows (launch_heavy_slots / launch_band_index), or null.
  // hslot[k] is row k's slot (-1: not banded); band + slot * nb1 are the slot's band positions.
  const int32_t* hslot = nullptr;
  const int32_t* band = nullptr;
  int64_t nb1 = 0;
  int64_t band_min = 0;  // smallest length of a banded row
};

// One category's kernel shape, chosen by the planner/autotuner.
struct KernelShape {
  int T;   // LDS hash slots (power of two); 0 = long-row window kernel; kHubShape = hub-row kernel
  int NT;  // threads per row group
  int G;   // lanes cooperating on one A entry (B row)
};
constexpr int kHubShape = -1;
// Hub rows: long rows whose output is computed in column ranges of kHubRange columns, one workgroup
// per (row, range). Of the rows of the long (last by key) category these are the ones with more
// than kHubEntries A entries (the windows of the other kernel visit them all, window after window)
// and the ones with at least per_range products for every range between their first and last
// column (kHubPerRange, so a range's products outweigh its clears, its emission and its visits of
// the entries).
#ifndef DBD_HUB_ENTRIES
#define DBD_HUB_ENTRIES 1024
#endif
#ifndef DBD_HUB_PER_RANGE
#define DBD_HUB_PER_RANGE 2048
#endif
constexpr int64_t kHubEntries = DBD_HUB_ENTRIES;
constexpr int64_t kHubPerRange = DBD_HUB_PER_RANGE;
constexpr int kHubRangeShift = 13;
constexpr int kHubRange = 1 << kHubRangeShift;
__host__ __device__ inline bool hub_row(int64_t nA, int64_t P, int nrng, int64_t per_range) {
  return nA > kHubEntries || P / nrng >= per_range;
}
// A slot value carries kHubMany for the rows of more than kHubEntries entries (plan reports count
// the others as long rows) and kHubFineBit for the rows counted range by range; a row's flag has a
// 1 for a hub row and a kHubFineOne for a fine one, so one scan gives its place in both lists.
constexpr int32_t kHubMany = 1 << 30, kHubFineBit = 1 << 29;
constexpr int32_t kHubSlotMask = kHubFineBit - 1;
constexpr int kHubFineShift = 40;
constexpr int64_t kHubFineOne = (int64_t)1 << kHubFineShift;

// ---- generic device utilities ----
void launch_fill_i64(int64_t* p, int64_t n, int64_t v, hipStream_t s);
void launch_fill_i32(int32_t* p, int64_t n, int32_t v, hipStream_t s);
void launch_fill_bytes0(void* p, int64_t nbytes, hipStream_t s);
// Exclusive scan of n int64 (in may equal out); out[n] = total. tmp needs scan_tmp_elems(n).
int64_t scan_tmp_elems(int64_t n);
void launch_exclusive_scan(const int64_t* in, int64_t* out, int64_t n, int64_t* tmp, hipStream_t s);
// Inside a captured pipeline: if *total > cap, set the capacity bit (16) in *err and zero
// offs[0 .. n), which empties every bin range that the following row kernels read.
constexpr int kErrCapacityBit = 16;
void launch_capacity_guard(const int64_t* total, int64_t cap, int64_t* offs, int64_t n, int* err, hipStream_t s);

// ---- band index of long B rows ----
// Columns per band; band index rows have band_count(ncols) entries (a multiple of kBandPad
// bands, so every aligned long-row window lies inside, plus one entry holding the row length).
constexpr int kBandShift = 12;
constexpr int kBandPad = 32;
int64_t band_count(int64_t ncols);
constexpr int64_t kRankShort = 64;  // k_numeric_rank takes long rows if the index has all B rows from here on
// hist[j] (32 int64) = number of B rows with at least 2^j entries.
void launch_len_hist(const int64_t* Bptr, int64_t nrows, int64_t* hist, hipStream_t s);
// slot[k] = index of B row k among the rows of at least minlen entries (-1 for the others),
// slot_row[s] = the row of slot s. flag (nrows + 1 int64) and tmp (scan_tmp_elems(nrows + 1)) are
// scratch; flag[nrows] receives the number of slots.
void launch_heavy_slots(const int64_t* Bptr, int64_t nrows, int64_t minlen, int64_t* flag, int64_t* tmp,
                        int32_t* slot, int32_t* slot_row, hipStream_t s);
// band[s * nb1 + b] = position (from the row start) of slot s's first entry with column >= b * 4096;
// band[s * nb1 + nb1 - 1] = the row's length.
void launch_band_index(const int32_t* slot_row, int64_t nslots, const int64_t* Bptr, const int32_t* Bidx, int64_t nb1,
                       int32_t* band, hipStream_t s);

// ---- planning ----
// P[i] = sum_{k in A_i} len(B_k), nnz[i] = 0 and *err = 0; per A nonzero j with column k:
// bstart[j] = B.ptr[k], blen[j] = len(B_k). tile_row: scratch of row_tiles(nnz(A)) + 1 entries.
int64_t row_tiles(int64_t nnz);
void launch_row_products(const Mat& A, const Mat& B, int64_t* P, int64_t* nnz, int64_t* bstart, int32_t* blen,
                         int32_t* tile_row, int* err, hipStream_t s);
// Host memory (pinned) that the kernels report to; read it after synchronising the stream.
struct HostReport {
  int64_t tot[kMaxCats + 1];  // first row of every category in the list, the last: all rows
  int32_t err[2];             // error word; hub rows of many entries
  int64_t blk[1];             // per block the keys' sum before it; behind the last block the total
};
// Where a binning writes besides the list: the keys' exclusive prefix (n + 1 entries, twice if asked
// for) and a report with blocks of `bt` tiles. All optional (host null: no report).
struct BinOut {
  int64_t *ptr = nullptr, *ptr2 = nullptr;
  HostReport* host = nullptr;
  const int* err = nullptr;
  int64_t bt = 1;
};
// Stable counting sort of rows [0, n) by category of min(key[i], cap) into rows; offs (cat-major by
// tile of bin_tiles(n), then the number of rows plus the keys' prefix by tile) has (ct.n + 1) *
// bin_tiles(n) + 1 entries, counts (scratch) (ct.n + 1) * bin_tiles(n).
// With hub_slot, rows of the category before the last (the long one by key) that have a hub slot
// (>= 0) go to the last category (the hub category); *many counts those marked kHubMany.
int64_t bin_tiles(int64_t n);
void launch_bin(const int64_t* key, int64_t n, int64_t cap, const CatTable& ct, int64_t* counts, int64_t* offs,
                int64_t* tmp, int32_t* rows, const BinOut& o, hipStream_t s, const int32_t* hub_slot = nullptr,
                int* many = nullptr);
void launch_report_err(const int* err, HostReport* host, hipStream_t s);

// ---- symbolic / numeric / backward per category ----
// grid == 0 -> exact grid from nrows_hint, the number of rows; else a persistent grid of that many
// workgroups, nrows_hint a bound on the rows.
int symbolic_groups_per_wg(const KernelShape& k);
// With hub_slot, the long-row kernel leaves out the rows that have a slot (>= 0): launch_hub_count's.
void launch_symbolic(const KernelShape& k, const int32_t* rows, const int64_t* pbeg, const int64_t* pend,
                     int64_t nrows_hint, int grid, const Mat& A, const Mat& B, int64_t* nnz, int64_t* cursor,
                     int* err, hipStream_t s, const int32_t* hub_slot = nullptr);
// distinct: most products of the problem are distinct columns of their row (nnzC close to the
// product count); the one-wave shapes then take rows whose products are all distinct through a
// register path instead of the hash table.
void launch_numeric(int dtype, const KernelShape& k, const int32_t* rows, const int64_t* pbeg,
                    const int64_t* pend, int64_t nrows_hint, int grid, const Mat& A, const Mat& B,
                    const int64_t* Cptr, int64_t cbase, int32_t* Cidx, void* Cval, int64_t* cursor, int* err,
                    hipStream_t s, bool distinct = false);
// ---- hub rows ----
constexpr int kHubMaxRanges = 8192;
int hub_ranges(int64_t ncols);
// Ranges per window of the hub rows' symbolic count, for B of this width and so many long rows.
int hub_wide(int64_t ncols, int64_t nlong);
// Whether the short entries' products are bucketed per (row, range) for B of this width.
bool hub_buckets_used(int64_t ncols);
// Device workspace of the hub rows: their list (slot -> row) and slots (row -> slot, -1: none), the
// slots of the fine rows (counted range by range), chunk offsets of the split and the buckets
// (n + 1), scan partials, the entry records (16 bytes per A nonzero), per slot the number of banded
// and short entries and the column span (2), the columns per (slot, range), and what the range
// workgroups read of their row.
struct HubWork {
  int64_t n = 0, nfine = 0;
  int wide = 16;  // ranges per count window (hub_wide)
  int32_t *rows = nullptr, *slot = nullptr, *fine = nullptr, *hcnt = nullptr, *lcnt = nullptr, *span = nullptr,
          *rng_cnt = nullptr;
  int64_t *coff = nullptr, *boff = nullptr, *tmp = nullptr;
  void *recs = nullptr, *info = nullptr;
};
constexpr size_t kHubRowBytes = 32;  // of info, per row of a chunk
// flag[j] of rows[j] by hub_row; with pos the exclusive scan of flag: h's slots (filled with -1
// first), list and fine list.
void launch_hub_flags(const int32_t* rows, int64_t n, const Mat& A, const Mat& B, const int64_t* P, int64_t per_range,
                      int wide, int64_t products, int64_t* flag, hipStream_t s);
void launch_hub_slots(const int32_t* rows, int64_t n, const Mat& A, const int64_t* flag, const int64_t* pos,
                      const HubWork& h, hipStream_t s);
// The rows' entries by kind into h.recs (hcnt, lcnt, span), nnz of the rows and *many cleared. Rows that are
// not long by their products (min(P, ncols) <= key_lim) are left empty.
void launch_hub_split(const HubWork& h, const Mat& A, const Mat& B, const int64_t* P, int64_t key_lim, int64_t* nnz,
                      int* many, hipStream_t s);
// Columns per (slot, range) into h.rng_cnt, their sums added to nnz (after launch_hub_split).
void launch_hub_count(const HubWork& h, const Mat& A, const Mat& B, int64_t* nnz, hipStream_t s);
// For the hub rows rows[0, n) of a chunk. gather: rcnt[j * nrng + r] = the row's columns per range,
// and h.info. bucket_count: short entries' products per (row, range) into scnt[n * nrng];
// bucket_fill: those products, (column, value), at soff (the exclusive scan of scnt; scnt is used
// up). guard: sets the capacity bit in err when *total short products exceed cap, on which
// bucket_fill and range write nothing. range: the values, emitted at Cptr[row] - cbase + roff[item]
// - roff[row's first item]; soff null: no buckets, the short entries are read from B.
void launch_hub_gather_counts(const HubWork& h, const int32_t* rows, int64_t n, const Mat& A, const Mat& B,
                              const int64_t* Cptr, int64_t cbase, int64_t* rcnt, hipStream_t s);
void launch_hub_bucket_count(const HubWork& h, const int32_t* rows, int64_t n, const Mat& A, const Mat& B,
                             int64_t* scnt, hipStream_t s);
void launch_hub_bucket_fill(int dtype, const HubWork& h, const int32_t* rows, int64_t n, const Mat& A, const Mat& B,
                            int64_t* scnt, const int64_t* soff, int32_t* scol, void* sval, const int* err,
                            hipStream_t s);
void launch_hub_guard(const int64_t* total, int64_t cap, int* err, hipStream_t s);
void launch_hub_range(int dtype, const HubWork& h, int64_t nh, const Mat& A, const Mat& B, const int64_t* soff,
                      const int32_t* scol, const void* sval, const int64_t* roff, int32_t* Cidx, void* Cval, int* err,
                      hipStream_t s);

// Gradients of the hub rows (their columns per range gathered and scanned as for range, with the
// caller's Cptr and cbase 0); dA is 0 beforehand. hub_backward_ranges: 0 if B is too wide for it.
int hub_backward_ranges(int dtype, int64_t ncols);
void launch_hub_backward(int dtype, const HubWork& h, int64_t n, const Mat& A, const Mat& B, const int64_t* roff,
                         const int32_t* Cidx, const void* dC, void* dA, void* dB, int64_t db_stride, int* err, hipStream_t s);

// dB's products go to dB + (part) * db_stride: 0 for dB itself, nnz(B) for a workspace of
// db_part_bytes (0: none is wanted) cleared beforehand, which launch_db_sum adds to dB.
size_t db_part_bytes(int dtype, int64_t products, int64_t nnzB);
void launch_db_sum(const void* part, int64_t n, void* dB, hipStream_t s);
void launch_backward(int dtype, const KernelShape& k, const int32_t* rows, const int64_t* pbeg,
                     const int64_t* pend, int64_t nrows_hint, int grid, const Mat& A, const Mat& B,
                     const int64_t* Cptr, const int32_t* Cidx, const void* dC, void* dA, void* dB, int64_t db_stride, int64_t* cursor,
                     int* err, hipStream_t s);
// Is this (T, NT, G) compiled? (the autotuner only proposes compiled shapes)
bool shape_available(int phase, const KernelShape& k);  // phase 0 symbolic, 1 numeric, 2 backward

}  // namespace dbd
