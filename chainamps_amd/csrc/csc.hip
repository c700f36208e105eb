// CSC form of a block tensor, sorted on the device.
//
// A block's rows (its first `numrows` indices) and columns are Cartesian
// products of sectors, and in block storage its rows come first.  So every
// column of one column-sector tuple (a class) holds the same rows, and its
// entries stand at base + coloff * stride with base and stride per row and
// coloff per column.  The host lists each class's rows once, in ascending
// order; two passes with one workgroup per column then count and compact the
// nonzero entries in place of a sort over all of them.
#include <algorithm>
#include <unordered_map>

#include "bstensor.hpp"

namespace cam {

namespace {

struct CscRow {
  int64_t row, base, stride;
};
struct CscCol {
  int64_t off;           // column within its sector tuple
  int32_t first, count;  // its class's rows
};

constexpr int kCscThreads = 256;

// Position of this thread's entry among the kept ones of the workgroup's
// chunk; `total` gets their number.
__device__ __forceinline__ int chunk_position(bool keep, int* wave_count, int& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long mask = __ballot(keep);
  if (lane == 0) wave_count[wave] = __popcll(mask);
  __syncthreads();
  int before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < kCscThreads / 64; ++w) {
    if (w < wave) before += wave_count[w];
    total += wave_count[w];
  }
  __syncthreads();
  return before + __popcll(mask & ((1ull << lane) - 1ull));
}

// Count (row and x null) or emission of the nonzero entries of columns
// c0 + blockIdx.x ...: bound by one read of the blocks (rows of a class are
// runs of consecutive elements) and, for the emission, 24 bytes written per
// entry and their copy to the host.
__global__ __launch_bounds__(kCscThreads) void csc_kernel(const double2* __restrict__ data,
                                                          const CscCol* __restrict__ cols,
                                                          const CscRow* __restrict__ rows, int64_t c0, int64_t c1,
                                                          int64_t* __restrict__ count, const int64_t* __restrict__ start,
                                                          int64_t* __restrict__ row, double2* __restrict__ x) {
  __shared__ int wave_count[kCscThreads / 64];
  for (int64_t c = c0 + blockIdx.x; c < c1; c += gridDim.x) {
    const CscCol C = cols[c];
    int64_t done = 0;
    for (int r0 = 0; r0 < C.count; r0 += kCscThreads) {
      const int r = r0 + static_cast<int>(threadIdx.x);
      CscRow R{};
      double2 v = make_double2(0.0, 0.0);
      if (r < C.count) {
        R = rows[C.first + r];
        v = data[R.base + C.off * R.stride];
      }
      const bool keep = r < C.count && !(v.x == 0.0 && v.y == 0.0);
      int total;
      const int pos = chunk_position(keep, wave_count, total);
      if (row && keep) {
        const int64_t k = start[c] - start[c0] + done + pos;
        row[k] = R.row;
        x[k] = v;
      }
      done += total;
    }
    if (!row && threadIdx.x == 0) count[c] = done;
  }
}

}  // namespace

// At least kCscElements elements, and class tables an eighth of them at most
// (a tensor with few columns has as many table rows as entries, which the host
// would have to sort all the same).
// Both routes, two calls (count, fill) each, random tensors with 2-9 sectors
// per index: 8192 elements 263 us on the host, 260 here; 32768 909 us and 404;
// 131072 4.8 ms and 0.41; 295000 9.9 ms and 0.49.
static constexpr int64_t kCscElements = 16384;
static constexpr int64_t kCscChunk = int64_t(1) << 22;   // entries emitted at a time (24 bytes each)

bool tensor_to_csc_device(const BSTensor& t, int64_t cap, int64_t* p, int64_t* ii, double* x, hipStream_t s,
                          int64_t& nnz) {
  if (t.total < kCscElements) return false;
  const int n = t.nidx(), nr = t.numrows;
  const int64_t ncols = t.cols();
  std::vector<int64_t> stride(n);
  int64_t m = 1;
  for (int k = 0; k < n; ++k) {
    if (k == nr) m = 1;
    stride[k] = m;
    m *= t.idx[k].size;
  }
  auto product = [](const Block& b, int lo, int hi) {
    int64_t q = 1;
    for (int k = lo; k < hi; ++k) q *= b.dims[k];
    return q;
  };
  int64_t table = 0;
  for (const Block& b : t.blocks) table += product(b, 0, nr);
  if (table > t.total / 8 || ncols > t.total / 8) return false;
  // classes: blocks of one column-sector tuple
  struct Class { std::vector<const Block*> blocks; };
  std::vector<Class> classes;
  std::unordered_map<uint64_t, int> class_of;
  auto col_code = [&](const Block& b) {
    uint64_t code = 0, mult = 1;
    for (int k = nr; k < n; ++k) {
      code += static_cast<uint64_t>(b.sec[k]) * mult;
      mult *= static_cast<uint64_t>(std::max(1, t.idx[k].nsec()));
    }
    return code;
  };
  for (const Block& b : t.blocks) {
    if (!b.size) continue;
    auto it = class_of.emplace(col_code(b), static_cast<int>(classes.size())).first;
    if (it->second == static_cast<int>(classes.size())) classes.emplace_back();
    classes[it->second].blocks.push_back(&b);
  }
  std::vector<CscRow> rows;
  rows.reserve(static_cast<size_t>(table));
  std::vector<CscCol> cols(static_cast<size_t>(ncols), CscCol{0, 0, 0});
  std::vector<int64_t> at(n);
  for (const Class& cl : classes) {
    const size_t first = rows.size();
    for (const Block* b : cl.blocks) {
      const int64_t R = product(*b, 0, nr);
      std::fill(at.begin(), at.end(), 0);
      for (int64_t r = 0; r < R; ++r) {
        int64_t pos = 0;
        for (int k = 0; k < nr; ++k) pos += t.idx[k].sec_pos[b->sec[k]][at[k]] * stride[k];
        rows.push_back(CscRow{pos, b->offset + r, R});
        for (int k = 0; k < nr && ++at[k] == b->dims[k]; ++k) at[k] = 0;
      }
    }
    std::sort(rows.begin() + first, rows.end(), [](const CscRow& a, const CscRow& b) { return a.row < b.row; });
    const Block& b0 = *cl.blocks.front();
    const int64_t C = product(b0, nr, n);
    std::fill(at.begin(), at.end(), 0);
    for (int64_t c = 0; c < C; ++c) {
      int64_t pos = 0;
      for (int k = nr; k < n; ++k) pos += t.idx[k].sec_pos[b0.sec[k]][at[k]] * stride[k];
      cols[static_cast<size_t>(pos)] = CscCol{c, static_cast<int32_t>(first), static_cast<int32_t>(rows.size() - first)};
      for (int k = nr; k < n && ++at[k] == b0.dims[k]; ++k) at[k] = 0;
    }
  }
  if (rows.size() > (size_t(1) << 30)) return false;
  // without room on the device the host does it
  auto room = [](auto& buf, size_t count) {
    try {
      buf.alloc(count);
    } catch (const Error&) {
      (void)hipGetLastError();
      return false;
    }
    return true;
  };
  DevBuf<CscRow> drows;
  DevBuf<CscCol> dcols;
  DevBuf<int64_t> dstart;
  if (!room(drows, rows.size()) || !room(dcols, cols.size()) || !room(dstart, cols.size() + 1)) return false;
  drows.upload(rows.data(), rows.size(), s);
  dcols.upload(cols.data(), cols.size(), s);
  const double2* data = reinterpret_cast<const double2*>(t.data.get());
  auto grid = [](int64_t c) { return dim3(static_cast<unsigned>(std::min<int64_t>(c, 65536))); };
  hipLaunchKernelGGL(csc_kernel, grid(ncols), dim3(kCscThreads), 0, s, data, dcols.get(), drows.get(), int64_t(0),
                     ncols, dstart.get(), static_cast<const int64_t*>(nullptr), static_cast<int64_t*>(nullptr),
                     static_cast<double2*>(nullptr));
  HIP_CHECK(hipGetLastError());
  std::vector<int64_t> start(static_cast<size_t>(ncols) + 1, 0);
  HIP_CHECK(hipMemcpyAsync(start.data() + 1, dstart.get(), ncols * sizeof(int64_t), hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  for (int64_t c = 0; c < ncols; ++c) start[c + 1] += start[c];
  nnz = start[ncols];
  if (!p || nnz > cap) return true;
  // whole columns, as many as fit a chunk of entries (at least one)
  int64_t longest = 0;
  for (int64_t c = 0; c < ncols; ++c) longest = std::max(longest, start[c + 1] - start[c]);
  const int64_t chunk = std::min(nnz, std::max(kCscChunk, longest));
  DevBuf<int64_t> drow;
  DevBuf<cplx> dx;
  if (nnz && (!room(drow, chunk) || !room(dx, chunk))) return false;
  std::copy(start.begin(), start.end(), p);
  dstart.upload(start.data(), start.size(), s);
  for (int64_t c0 = 0; c0 < ncols && nnz;) {
    int64_t c1 = c0 + 1;
    while (c1 < ncols && start[c1 + 1] - start[c0] <= chunk) ++c1;
    const int64_t k = start[c1] - start[c0];
    if (k) {
      hipLaunchKernelGGL(csc_kernel, grid(c1 - c0), dim3(kCscThreads), 0, s, data, dcols.get(), drows.get(), c0, c1,
                         static_cast<int64_t*>(nullptr), static_cast<const int64_t*>(dstart.get()), drow.get(),
                         reinterpret_cast<double2*>(dx.get()));
      HIP_CHECK(hipGetLastError());
      HIP_CHECK(hipMemcpyAsync(ii + start[c0], drow.get(), k * sizeof(int64_t), hipMemcpyDeviceToHost, s));
      HIP_CHECK(hipMemcpyAsync(x + 2 * start[c0], dx.get(), k * sizeof(cplx), hipMemcpyDeviceToHost, s));
    }
    c0 = c1;
  }
  HIP_CHECK(hipStreamSynchronize(s));
  return true;
}

}  // namespace cam
