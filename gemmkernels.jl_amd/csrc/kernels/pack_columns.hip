// gk_pack_columns: the columns of one or two matrices of 16-bit elements, copied to a leading dimension that is a whole
// number of 128-byte lines.
//
// Bound by memory: a wave copies 1 KiB of a column with one 16-byte load per lane at whatever 2-byte alignment the column
// has and one aligned 16-byte store, four columns at a time so that four loads of a lane are in flight.  The chunk that reaches over the
// end of a column is loaded as the 16 bytes that end with it and shifted down, which brings in the zeros behind it.  Two operands of 32 MB take 24 us
// on the same inputs over and over, 25 on inputs that rotate through 256 MB (5.2 TB/s read and written; 33 where the end of a column went element by element).
#include "common.hpp"
#include "gk_internal.hpp"

namespace gk {
namespace {

struct PackJob {
  const unsigned short* src;
  unsigned short* dst;
  long long ld, ld_dst;
  long long rows, cols;
  long long rows_dst, cols_dst;      // of the copy: zero outside the matrix
  unsigned segments;                 // pieces of kPackRows rows of a column of the copy
};

constexpr int kPackCols = 4;                    // columns of a wave
constexpr int kPackWaves = 4;
constexpr int kPackRows = 8 * kWaveSize;        // rows of a wave

struct __attribute__((packed, aligned(2))) Chunk { int4v v; };

// A lane's chunk of 8 rows that reaches over the last row of a column: the 8 elements that end with the column, moved down by
// the `over` rows that lie outside, zeros behind them.
__device__ __forceinline__ int4v shifted_down(int4v x, int over) {
  const unsigned __int128 bits = __builtin_bit_cast(unsigned __int128, x);
  return __builtin_bit_cast(int4v, over < 8 ? bits >> (16 * over) : (unsigned __int128)0);
}

__global__ __launch_bounds__(kPackWaves * kWaveSize) void pack_columns_kernel(PackJob job0, PackJob job1, unsigned blocks0) {
  const bool second = blockIdx.x >= blocks0;
  const PackJob job = second ? job1 : job0;
  const unsigned block = blockIdx.x - (second ? blocks0 : 0), group = block / job.segments, segment = block - group * job.segments;
  const long long rows = job.rows, ld_dst = job.ld_dst;
  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const long long col0 = ((long long)group * kPackWaves + wave) * kPackCols;
  const long long row = (long long)segment * kPackRows + lane * 8;
  if (row >= job.rows_dst || col0 >= job.cols_dst) return;
  int4v x[kPackCols];
  if (rows >= 8) {
    const long long first = row < rows - 8 ? row : rows - 8;
    const int over = (int)(row - first < 8 ? row - first : 8);
#pragma unroll
    for (int i = 0; i < kPackCols; ++i)            // (columns past the last one: the last one again, not used)
      x[i] = ((const Chunk*)(job.src + (col0 + i < job.cols ? col0 + i : job.cols - 1) * job.ld + first))->v;
#pragma unroll
    for (int i = 0; i < kPackCols; ++i) {
      if (over != 0) x[i] = shifted_down(x[i], over);
      if (col0 + i >= job.cols) x[i] = int4v{0, 0, 0, 0};
    }
  } else {
#pragma unroll
    for (int i = 0; i < kPackCols; ++i) {
      unsigned e[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) e[r] = row + r < rows && col0 + i < job.cols ? job.src[(col0 + i) * job.ld + row + r] : 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) x[i][q] = (int)(e[2 * q] | e[2 * q + 1] << 16);
    }
  }
#pragma unroll
  for (int i = 0; i < kPackCols; ++i) {
    if (col0 + i >= job.cols_dst) continue;
    unsigned short* to = job.dst + (col0 + i) * ld_dst + row;
    if (row + 8 <= job.rows_dst) {
      *(int4v*)to = x[i];
    } else {
#pragma unroll
      for (int r = 0; r < 8; ++r)
        if (row + r < job.rows_dst) to[r] = (unsigned short)((unsigned)x[i][r / 2] >> (16 * (r % 2)));
    }
  }
}

int pack(PackJob (&jobs)[2], void* stream) {
  using gk_internal::fail;
  int64_t blocks[2] = {0, 0};
  for (int i = 0; i < 2; ++i) {
    PackJob& j = jobs[i];
    if (i == 1 && j.cols == 0) break;
    if (j.rows <= 0 || j.cols <= 0) return fail(GK_ERR_INVALID_ARGUMENT, "gk_pack_columns: sizes must be positive");
    if (!j.src || !j.dst) return fail(GK_ERR_INVALID_ARGUMENT, "gk_pack_columns: NULL pointer");
    if (j.rows_dst < j.rows || j.cols_dst < j.cols) return fail(GK_ERR_INVALID_ARGUMENT, "gk_pack_columns: a copy holds the matrix whole");
    if (j.ld < j.rows || j.ld_dst < j.rows_dst || j.ld_dst % 8 != 0)
      return fail(GK_ERR_INVALID_ARGUMENT, "gk_pack_columns: leading dimensions must hold a column, that of the copy in whole 16-byte vectors");
    if (((uintptr_t)j.src & 1u) != 0 || ((uintptr_t)j.dst & 15u) != 0)
      return fail(GK_ERR_ALIGNMENT, "gk_pack_columns: a matrix has 2-byte elements and its copy starts on a 16-byte boundary");
    const int64_t groups = (j.cols_dst - 1) / (kPackWaves * kPackCols) + 1, segments = (j.rows_dst - 1) / kPackRows + 1;
    if (groups > 0x7fffff || segments > 0xff) return fail(GK_ERR_INVALID_ARGUMENT, "gk_pack_columns: more columns or rows than one launch takes");
    j.segments = (unsigned)segments;
    blocks[i] = groups * segments;
  }
  if (blocks[0] + blocks[1] > 0x7fffffff) return fail(GK_ERR_INVALID_ARGUMENT, "gk_pack_columns: more columns or rows than one launch takes");
  hipLaunchKernelGGL(pack_columns_kernel, dim3((unsigned)(blocks[0] + blocks[1])), dim3(kPackWaves * kWaveSize), 0, (hipStream_t)stream, jobs[0], jobs[1],
                     (unsigned)blocks[0]);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(GK_ERR_HIP, "HIP launch of pack_columns failed: %s", hipGetErrorString(e));
  return GK_OK;
}

}  // namespace
}  // namespace gk

extern "C" {

int gk_pack_columns_padded(const void* src0, int64_t rows0, int64_t cols0, int64_t ld0, void* dst0, int64_t ld_dst0, int64_t rows_dst0, int64_t cols_dst0,
                           const void* src1, int64_t rows1, int64_t cols1, int64_t ld1, void* dst1, int64_t ld_dst1, int64_t rows_dst1, int64_t cols_dst1,
                           void* stream) {
  gk::PackJob jobs[2] = {{(const unsigned short*)src0, (unsigned short*)dst0, ld0, ld_dst0, rows0, cols0, rows_dst0, cols_dst0, 1},
                         {(const unsigned short*)src1, (unsigned short*)dst1, ld1, ld_dst1, rows1, cols1, rows_dst1, cols_dst1, 1}};
  return gk::pack(jobs, stream);
}

int gk_pack_columns(const void* src0, int64_t rows0, int64_t cols0, int64_t ld0, void* dst0, int64_t ld_dst0, const void* src1, int64_t rows1, int64_t cols1,
                    int64_t ld1, void* dst1, int64_t ld_dst1, void* stream) {
  return gk_pack_columns_padded(src0, rows0, cols0, ld0, dst0, ld_dst0, rows0, cols0, src1, rows1, cols1, ld1, dst1, ld_dst1, rows1, cols1, stream);
}

}  // extern "C"
