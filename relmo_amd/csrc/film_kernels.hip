// FiLM step of a central MLP with its Mish activation, fused:
//
//   y = mish(beta[k] + gamma[k] * (s + add[k]))   for the rows of range k,
//
// where the rows of one range share their gamma / beta / add rows (the rows of
// one predicate: the condition and the slot mask are constant per predicate).
// One pass over s replaces torch's add, addcmul, Mish and the concatenation of
// the per-range results; the backward reads s and the upstream gradient once,
// writes ds and leaves per-block column sums of du * (s + add) and du (du the
// gradient at the Mish input), in fp64, for the per-range gamma / beta
// gradients.
#include <hip/hip_runtime.h>

#include "device_utils.h"
#include "internal.h"

namespace relm_mp {

namespace {

constexpr int kThreads = 256;
constexpr int64_t kCus = 256;
constexpr int kMaxRanges = RELM_MP_FILM_MAX_RANGES;

// Range k covers rows [start[k], start[k + 1]); its blocks of rows_per_block
// rows are blocks [first_block[k], first_block[k + 1]), so no block spans two
// ranges.
struct FilmRanges {
    int64_t start[kMaxRanges + 1];
    int64_t first_block[kMaxRanges + 1];
    int64_t rows_per_block;
    int num;
};

// Mish and its derivative in the fp32 formulation of PyTorch's own Mish
// kernels (torch.nn.functional.mish and its backward on ROCm):
//   mish(u)         = u * tanh(log1p(exp(u)))
//   dy * mish'(u)   = dy * (t + u * sigmoid(u) * (1 - t * t)),  t = tanh(log1p(exp(u))),
// with the two multiply-adds of the derivative fused as torch's build fuses
// them, the accurate expf / log1pf / tanhf and IEEE division.  Together with
// the affine step b + g * (s + a) rounded as torch's addcmul rounds it, the
// fused step computes exactly what torch's FiLM and Mish ops compute, bit for
// bit (checked against them on the GPU).  The weight gradient of the Linear
// before the FiLM step is a sum over all rows with large cancellation; its
// rounding error moves by a factor of three with the last bit of a few rows'
// gradients, so a different (even more accurate) formulation leaves the
// models' gradients at a different fp32 error than the torch lane's.
// At u >= 10 that formulation has t = 1 exactly (log1p(exp(u)) > 10, whose
// tanh rounds to 1), so mish(u) = u and the gradient is dy; at u <= -104
// exp(u) is 0 in fp32, so t = 0: mish(u) = u * 0 and the gradient dy * +0.  The shortcuts
// skip the transcendental calls there and give the same bits (tested over
// dense sweeps of both ranges against torch).
constexpr float kMishOne = 10.0f;
constexpr float kMishZero = -104.0f;

__device__ __forceinline__ float mish(float u) {
    if (u >= kMishOne) return u;
    if (u <= kMishZero) return u * 0.0f;
    return u * tanhf(log1pf(expf(u)));
}

__device__ __forceinline__ float mish_backward(float dy, float u) {
    if (u >= kMishOne) return dy;
    if (u <= kMishZero) return dy * 0.0f;  // fma(u * 0, 1, 0) = +0 in the full formula
    const float sg = 1.0f / (1.0f + expf(-u));
    const float t = tanhf(log1pf(expf(u)));
    return dy * fmaf(u * sg, fmaf(-t, t, 1.0f), t);
}

// V floats that start at any 4-byte aligned address: one 16-byte access for V =
// 4, one of 8 for V = 2 (global memory takes them at dword alignment).
template <int V>
using Vec = float __attribute__((ext_vector_type(V), aligned(4)));

template <int V>
__device__ __forceinline__ Vec<V> load(const float* p) {
    return *reinterpret_cast<const Vec<V>*>(p);
}
template <int V>
__device__ __forceinline__ Vec<V> load_stream(const float* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const Vec<V>*>(p));
}
template <int V>
__device__ __forceinline__ void store_stream(float* p, Vec<V> x) {
    __builtin_nontemporal_store(x, reinterpret_cast<Vec<V>*>(p));
}

// A workgroup's rows and their range: blocks of a range are consecutive.
struct BlockRows {
    int k;
    int64_t r0;
    int64_t r1;
};

__device__ __forceinline__ BlockRows block_rows(const FilmRanges& R, int64_t b) {
    int k = 0;
#pragma unroll
    for (int q = 1; q < kMaxRanges; ++q)
        if (q < R.num && b >= R.first_block[q]) k = q;
    const int64_t r0 = R.start[k] + (b - R.first_block[k]) * R.rows_per_block;
    const int64_t r1 = min(r0 + R.rows_per_block, R.start[k + 1]);
    return {k, r0, r1};
}

// Thread layout of both kernels.  The columns are units of V floats; where the
// width is no multiple of V the last unit is shifted back to end with the row,
// and the columns it shares with the unit before are computed twice with equal
// results.  A workgroup takes `units` neighbouring units of one block of rows,
// `phases` rows at a time: thread t owns unit t % units and the block's rows t /
// units, t / units + phases, ...  A thread keeps its columns, so their tables
// stay in registers and the backward's column sums need no atomics.
struct FilmLayout {
    int total;   // units of a row
    int chunks;  // workgroups side by side over the columns
    int units;   // units of one workgroup
    int phases;  // rows of one workgroup at a time
};

struct FilmThread {
    int64_t col;
    int unit;
    int phase;
    bool active;
};

template <int V>
__device__ __forceinline__ FilmThread film_thread(const FilmLayout& L, int chunk, int64_t width) {
    const int t = static_cast<int>(threadIdx.x);
    FilmThread f;
    f.phase = t / L.units;
    f.unit = t - f.phase * L.units;
    const int u = chunk * L.units + f.unit;
    f.active = f.phase < L.phases && u < L.total;
    f.col = min(static_cast<int64_t>(u) * V, width - V);
    return f;
}

// Rows a thread has in flight: the loads of kRows rows are issued before the
// first of them is used.
constexpr int kRows = 2;

// Bound by the vector units, not by memory: 160 lane instructions per element
// (counted; most of them in expf, log1pf and tanhf), so 400 M elements take 1.2 ms
// at any split while moving them takes 0.64.  The workgroups are small (4 waves) and
// many, so that the last ones leave few CUs idle: [1,000,003 x 400] takes 1.34
// ms, [204,800 x 96] 76 us and [2,000 x 400] 10 us, against 1.46 ms, 86 us and
// 158 us with 768 threads to a workgroup of 512 whole rows.
template <int V>
__global__ __launch_bounds__(kThreads) void k_film_mish(const float* __restrict__ s, int64_t width,
                                                        FilmRanges R, FilmLayout L,
                                                        const float* __restrict__ gamma,
                                                        const float* __restrict__ beta,
                                                        const float* __restrict__ add,
                                                        float* __restrict__ y) {
    const int chunk = static_cast<int>(blockIdx.x % L.chunks);
    const BlockRows br = block_rows(R, blockIdx.x / L.chunks);
    const FilmThread f = film_thread<V>(L, chunk, width);
    if (!f.active) return;
    const Vec<V> g = load<V>(gamma + br.k * width + f.col);
    const Vec<V> b = load<V>(beta + br.k * width + f.col);
    const Vec<V> a = add != nullptr ? load<V>(add + br.k * width + f.col) : Vec<V>(0.0f);
    auto step = [&](const Vec<V>& x, int64_t r) {
        Vec<V> o;
#pragma unroll
        for (int i = 0; i < V; ++i) o[i] = mish(b[i] + g[i] * (x[i] + a[i]));
        store_stream<V>(y + r * width + f.col, o);
    };
    int64_t r = br.r0 + f.phase;
    for (; r + (kRows - 1) * L.phases < br.r1; r += kRows * L.phases) {
        Vec<V> x[kRows];
#pragma unroll
        for (int j = 0; j < kRows; ++j) x[j] = load_stream<V>(s + (r + j * L.phases) * width + f.col);
#pragma unroll
        for (int j = 0; j < kRows; ++j) step(x[j], r + j * L.phases);
    }
    for (; r < br.r1; r += L.phases) step(load_stream<V>(s + r * width + f.col), r);
}

// ds = dy * mish'(u) * gamma; partial[block][0][col] = sum over the block's
// rows of du * (s + add), partial[block][1][col] = sum of du, du = dy *
// mish'(u), each term rounded to fp32 and added in fp64: by each thread over
// its rows in row order, then the phases in order.  The block sums stay fp64
// (a range's blocks are added in fp64 and rounded once), so a per-range sum
// over tens of thousands of rows carries only the rounding of its terms.
// `lds` holds phases * units * V * 2 doubles.  Bound as the forward is (195 lane
// instructions per element): [1,000,003
// x 400] takes 1.67 ms with the sums, [204,800 x 96] 101 us, against 2.18 ms and
// 134 us with the forward's former split and torch's sums.
template <int V>
__global__ __launch_bounds__(kThreads) void k_film_mish_backward(
    const float* __restrict__ s, const float* __restrict__ dy, int64_t width, FilmRanges R,
    FilmLayout L, const float* __restrict__ gamma, const float* __restrict__ beta,
    const float* __restrict__ add, float* __restrict__ ds, double* __restrict__ partial) {
    extern __shared__ double lds[];
    const int chunk = static_cast<int>(blockIdx.x % L.chunks);
    const int64_t block = blockIdx.x / L.chunks;
    const BlockRows br = block_rows(R, block);
    const FilmThread f = film_thread<V>(L, chunk, width);
    if (f.active) {
        const Vec<V> g = load<V>(gamma + br.k * width + f.col);
        const Vec<V> b = load<V>(beta + br.k * width + f.col);
        const Vec<V> a = add != nullptr ? load<V>(add + br.k * width + f.col) : Vec<V>(0.0f);
        double sum_t[V], sum_u[V];
#pragma unroll
        for (int i = 0; i < V; ++i) sum_t[i] = sum_u[i] = 0.0;
        auto step = [&](const Vec<V>& x, const Vec<V>& d, int64_t r) {
            Vec<V> o;
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const float tt = x[i] + a[i];
                const float du = mish_backward(d[i], b[i] + g[i] * tt);
                o[i] = du * g[i];
                sum_t[i] += static_cast<double>(du * tt);
                sum_u[i] += static_cast<double>(du);
            }
            store_stream<V>(ds + r * width + f.col, o);
        };
        int64_t r = br.r0 + f.phase;
        for (; r + (kRows - 1) * L.phases < br.r1; r += kRows * L.phases) {
            Vec<V> x[kRows], d[kRows];
#pragma unroll
            for (int j = 0; j < kRows; ++j) {
                x[j] = load_stream<V>(s + (r + j * L.phases) * width + f.col);
                d[j] = load_stream<V>(dy + (r + j * L.phases) * width + f.col);
            }
#pragma unroll
            for (int j = 0; j < kRows; ++j) step(x[j], d[j], r + j * L.phases);
        }
        for (; r < br.r1; r += L.phases)
            step(load_stream<V>(s + r * width + f.col), load_stream<V>(dy + r * width + f.col), r);
        // this thread's sums into LDS: [phase][t or u][unit][V]
        double* l = lds + (static_cast<int64_t>(f.phase) * 2 * L.units + f.unit) * V;
#pragma unroll
        for (int i = 0; i < V; ++i) {
            l[i] = sum_t[i];
            l[L.units * V + i] = sum_u[i];
        }
    }
    __syncthreads();
    // one thread per (t or u, column) adds the phases in order
    const int sums = 2 * L.units * V;
    for (int i = static_cast<int>(threadIdx.x); i < sums; i += kThreads) {
        const int which = i / (L.units * V), at = i - which * (L.units * V);
        const int u = chunk * L.units + at / V;
        if (u >= L.total) continue;
        double sum = 0.0;
        for (int p = 0; p < L.phases; ++p) sum += lds[static_cast<int64_t>(p) * sums + i];
        const int64_t col = min(static_cast<int64_t>(u) * V, width - V) + at % V;
        partial[(block * 2 + which) * width + col] = sum;
    }
}

// sums[k][j] = sum over range k's blocks of partial[block][j] (j < 2 * width),
// added in fp64 and rounded to fp32 once: kFoldCols columns by kFoldRows blocks
// at a time, then the kFoldRows parts in order.  Latency bound (at most a few
// tens of MB over many short chains): torch's sum took 16 us per range and a
// copy each.
constexpr int kFoldCols = 16;
constexpr int kFoldRows = kThreads / kFoldCols;

__global__ __launch_bounds__(kThreads) void k_film_fold(const double* __restrict__ partial, int64_t cols,
                                                        FilmRanges R, float* __restrict__ sums) {
    __shared__ double lds[kFoldRows][kFoldCols];
    const int c = static_cast<int>(threadIdx.x) % kFoldCols, q = static_cast<int>(threadIdx.x) / kFoldCols;
    const int k = static_cast<int>(blockIdx.y);
    const int64_t j = static_cast<int64_t>(blockIdx.x) * kFoldCols + c;
    double sum = 0.0;
    if (j < cols) {
        const int64_t b1 = R.first_block[k + 1];
        int64_t b = R.first_block[k] + q;
        for (; b + 3 * kFoldRows < b1; b += 4 * kFoldRows) {
            double v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = partial[(b + i * kFoldRows) * cols + j];
#pragma unroll
            for (int i = 0; i < 4; ++i) sum += v[i];
        }
        for (; b < b1; b += kFoldRows) sum += partial[b * cols + j];
    }
    lds[q][c] = sum;
    __syncthreads();
    if (q == 0 && j < cols) {
        for (int i = 1; i < kFoldRows; ++i) sum += lds[i][c];
        sums[k * cols + j] = static_cast<float>(sum);
    }
}

FilmRanges film_ranges(const int64_t* range_start, int32_t num_ranges, int64_t rows_per_block) {
    FilmRanges R{};
    int64_t blocks = 0;
    for (int k = 0; k < num_ranges; ++k) {
        R.start[k] = range_start[k];
        R.first_block[k] = blocks;
        blocks += film_range_blocks(range_start[k + 1] - range_start[k], rows_per_block);
    }
    for (int k = num_ranges; k <= kMaxRanges; ++k) {
        R.start[k] = range_start[num_ranges];
        R.first_block[k] = blocks;
    }
    R.rows_per_block = rows_per_block;
    R.num = num_ranges;
    return R;
}

// Units of a workgroup: all of a row's up to 64 (1 KB of a row with 16-byte
// units), else an even split of the row into chunks of at most 64, so that no
// chunk is nearly empty (100 units: 2 chunks of 50, 5 phases each, 250 of 256
// threads busy).
FilmLayout film_layout(int64_t width, int V) {
    const int64_t total = (width + V - 1) / V;
    FilmLayout L{static_cast<int>(total), static_cast<int>((total + 63) / 64), 0, 0};
    L.units = static_cast<int>((total + L.chunks - 1) / L.chunks);
    L.phases = kThreads / L.units;
    return L;
}

// Rows of a workgroup: from `least` to `most` per thread, as many as leave four
// workgroups to every CU.
int64_t film_rows_per_block(const FilmLayout& L, int64_t rows, int least, int most) {
    int per_thread = most;
    while (per_thread > least && rows * L.chunks < 4 * kCus * per_thread * L.phases) per_thread /= 2;
    return static_cast<int64_t>(per_thread) * L.phases;
}

// Floats of a unit: 4 at any alignment where they divide the row or the columns
// that the last unit computes twice are few (from 64 on), else 2.  In units of 4
// the forward of 67 M floats takes 287 us at width 6 and 252 at 10, the backward 459
// at 5 and 404 at 6; in units of 2 213, 208, 339 and 308 (227, 238, 407 and 361 by
// rows of whole 8- or 4-byte lanes in larger workgroups); at 201 and 398 the forward
// 269 and 238 us against 285 and 243.  3 floats go one by one (backward 305 us, 368
// in units of 2).  Where the output takes the place of an input, units that share no
// column: one must not be read again after another thread has written it.
int film_vec(int64_t width, bool in_place = false) {
    const int V = width % 4 == 0 || width >= 64 ? 4 : width == 1 || width == 3 ? 1 : 2;
    if (in_place && width % V != 0) return width % 2 == 0 ? 2 : 1;
    return V;
}

hipError_t film_backward(const float* s, const float* dy, int64_t width, const FilmRanges& R,
                         const float* gamma, const float* beta, const float* add, float* ds,
                         double* partial, hipStream_t st) {
    const int V = film_vec(width, ds == s || ds == dy);
    const FilmLayout L = film_layout(width, V);
    const dim3 grid(static_cast<unsigned>(R.first_block[kMaxRanges] * L.chunks));
    const size_t lds = static_cast<size_t>(L.phases) * L.units * V * 2 * sizeof(double);
    const auto kernel = V == 4   ? k_film_mish_backward<4>
                        : V == 2 ? k_film_mish_backward<2>
                                 : k_film_mish_backward<1>;
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), lds, st, s, dy, width, R, L, gamma, beta, add, ds, partial);
    return hipGetLastError();
}

// The split of relm_mp_film_mish_backward_sums: 8 to 64 rows per thread (the
// blocks' sums are read again, 16 bytes per column and block).
int64_t film_backward_rows(int64_t width, int64_t rows) {
    return film_rows_per_block(film_layout(width, film_vec(width)), rows, 8, 64);
}

}  // namespace

hipError_t launch_film_mish(const float* s, int64_t width, const int64_t* range_start,
                            int32_t num_ranges, const float* gamma, const float* beta,
                            const float* add, float* y, hipStream_t st) {
    const int64_t rows = range_start[num_ranges];
    if (rows == 0 || width == 0) return hipSuccess;
    const int V = film_vec(width, y == s);
    const FilmLayout L = film_layout(width, V);
    const FilmRanges R = film_ranges(range_start, num_ranges, film_rows_per_block(L, rows, 4, 16));
    const dim3 grid(static_cast<unsigned>(R.first_block[kMaxRanges] * L.chunks));
    const auto kernel = V == 4 ? k_film_mish<4> : V == 2 ? k_film_mish<2> : k_film_mish<1>;
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, st, s, width, R, L, gamma, beta, add, y);
    return hipGetLastError();
}

hipError_t launch_film_mish_backward(const float* s, const float* dy, int64_t width,
                                     const int64_t* range_start, int32_t num_ranges,
                                     const float* gamma, const float* beta, const float* add,
                                     float* ds, double* partial, hipStream_t st) {
    if (range_start[num_ranges] == 0 || width == 0) return hipSuccess;
    const FilmRanges R = film_ranges(range_start, num_ranges, RELM_MP_FILM_ROWS_PER_BLOCK);
    return film_backward(s, dy, width, R, gamma, beta, add, ds, partial, st);
}

size_t film_sums_workspace(const int64_t* range_start, int32_t num_ranges, int64_t width) {
    if (range_start[num_ranges] == 0 || width == 0) return 0;
    const FilmRanges R = film_ranges(range_start, num_ranges, film_backward_rows(width, range_start[num_ranges]));
    return static_cast<size_t>(R.first_block[kMaxRanges]) * 2 * width * sizeof(double);
}

hipError_t launch_film_mish_backward_sums(const float* s, const float* dy, int64_t width,
                                          const int64_t* range_start, int32_t num_ranges,
                                          const float* gamma, const float* beta, const float* add,
                                          float* ds, float* sums, double* partial, hipStream_t st) {
    if (width == 0) return hipSuccess;
    const int64_t rows = range_start[num_ranges];
    const FilmRanges R = film_ranges(range_start, num_ranges, film_backward_rows(width, rows));
    if (rows > 0) {
        const hipError_t e = film_backward(s, dy, width, R, gamma, beta, add, ds, partial, st);
        if (e != hipSuccess) return e;
    }
    const int64_t cols = 2 * width;
    hipLaunchKernelGGL(k_film_fold, dim3(static_cast<unsigned>((cols + kFoldCols - 1) / kFoldCols), num_ranges),
                       dim3(kThreads), 0, st, partial, cols, R, sums);
    return hipGetLastError();
}

}  // namespace relm_mp
