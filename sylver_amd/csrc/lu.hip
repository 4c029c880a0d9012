// Dense front LU of the unsymmetric path, batched on the device: the
// reference's kernels lu_nopiv_factor (src/kernels/lu_nopiv.hxx:13-41),
// lu_pp_factor (src/kernels/lu_pp.hxx:38-73) and lu_tpp_factor
// (src/kernels/lu_tpp.hxx:33-118) over many fronts in one launch.
//
// The front is held in registers: a row to a lane (two rows for orders over
// 64), the columns dealt to the W waves of its workgroup (column j to wave
// j mod W). Step e: the wave that holds the pivot column searches it, forms
// d = 1 / a_ee and l = a_ie d for the rows below, and hands l and the pivot
// row on through LDS; after one barrier every wave updates its own columns,
// a_ij = fma(-l, a_ej, a_ij), with a_ej read from the pivot row's lane. Rows
// and columns are never moved: each lane keeps its rows' positions, a pivot
// search takes the largest |a_ic| and on ties the row in the smaller position
// (the reference's find_col_abs_max, include/sylver/kernels/common.hxx:63-104,
// keeps the first row reaching the maximum), and the interchanges happen in
// the final store. The arithmetic and its order per entry are those of the
// CPU restatement in the oracle, so the factors agree bit for bit.
//
// Bound: the chain of steps (search, reciprocal, hand-over, update: about a
// thousand cycles at order 128), hidden by the other fronts on the CU. The
// form before, with the front in LDS and a thread per row, read and wrote
// every trailing entry there in each step and held one FP64 front per CU.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <vector>

#include "numeric.hpp"
#include "wave_ops.hpp"

namespace sylver_amd {

namespace {

constexpr int kLuMaxRows = 128;

struct LuTask {
   int64_t off;   // the front's first element in the caller's buffer (ld = m)
   int m, k;      // order and columns to eliminate
   int64_t perm;  // offset of the front's rperm / cperm entries
   int front, pad;
};

template <typename T>
__device__ inline T lu_abs(T v) {
   return v < T(0) ? -v : v;
}

// The columns of a wave, one register (pair) per column and row set: vectors,
// so that a column picked by a uniform index is an indexed register access
// (at most 32 dwords each) and the rest stays in registers.
template <typename T, int N>
using Cols = T __attribute__((ext_vector_type(N)));

// One front of order at most 64 S and at most W NC per workgroup of W waves.
template <typename T, int W, int S, int NC>
__global__ __launch_bounds__(64 * W, W >= 8 ? 4 : 1) void k_lu_front(const LuTask* __restrict__ tasks, T* __restrict__ data, int mode,
                                                     double u, int* __restrict__ rperm, int* __restrict__ cperm,
                                                     int* __restrict__ nelim_out) {
   __shared__ T lbuf[2][64 * S];         // l of a step, by row
   __shared__ int ctrl[2];               // its pivot row (-1: the candidate column was refused)
   __shared__ int colat[64 * S], posof[64 * S];  // physical column at each position, position of each column
   const LuTask t = tasks[blockIdx.x];
   const int m = t.m, k = t.k;
   T* F = data + t.off;
   const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   // position of each of the lane's rows (row lane + 64 s); -1: no such row
   int pos[S];
#pragma unroll
   for (int s = 0; s < S; ++s) pos[s] = lane + 64 * s < m ? lane + 64 * s : -1;
   constexpr int VL = NC < 16 ? NC : 16, H = NC / VL;
   Cols<T, VL> a[H][S];
#pragma unroll
   for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int s = 0; s < S; ++s) {
         const int j = c * W + wave;
         a[c / VL][s][c % VL] = (j < m && pos[s] >= 0) ? F[pos[s] + (int64_t)j * m] : T(0);
      }
   unsigned live = 0;  // columns of this wave not yet eliminated
#pragma unroll
   for (int c = 0; c < NC; ++c) live |= (c * W + wave < m ? 1u : 0u) << c;
   for (int j = threadIdx.x; j < m; j += 64 * W) colat[j] = j;
   __syncthreads();
   const T tu = T(u);
   int nelim = 0;
   // one candidate column per round: position c (modes 0 and 1: c = nelim)
   for (int c = 0, round = 0; c < k; ++round) {
      const int q = mode == 2 ? __builtin_amdgcn_readfirstlane(colat[c]) : c;  // physical column
      const int owner = q % W, cc = q / W, par = round & 1;
      T l[S];
      int prow = -1;
      if (wave == owner) {
         T x[S];
#pragma unroll
         for (int s = 0; s < S; ++s) x[s] = H == 1 || cc < VL ? a[0][s][cc % VL] : a[H - 1][s][cc % VL];
         // the row with the largest |x| among positions [nelim, to], the smaller position on ties
         auto abs_max = [&](int to, T& val) {
            T v[S], vm = T(-1);
#pragma unroll
            for (int s = 0; s < S; ++s) {
               v[s] = (pos[s] >= nelim && pos[s] <= to) ? lu_abs(x[s]) : T(-1);
               vm = v[s] > vm ? v[s] : vm;
            }
            val = wave_reduce(vm, [](T p, T r) { return r > p ? r : p; });
            int at = 0x7fffffff;
#pragma unroll
            for (int s = 0; s < S; ++s)
               if (pos[s] >= nelim && pos[s] <= to && v[s] == val) at = min(at, pos[s]);
            const unsigned long long hit = __ballot(at != 0x7fffffff);
            // one lane (and, of its rows, the smaller position), or the smallest position of several
            const int best = __builtin_popcountll(hit) == 1
                                 ? lane_value(at, __builtin_ctzll(hit))
                                 : wave_reduce(at, [](int p, int r) { return min(p, r); });
            return best;
         };
         // the row (lane + 64 s) at a position
         auto row_at = [&](int position) {
            int row = 0;
#pragma unroll
            for (int s = 0; s < S; ++s) {
               const unsigned long long b = __ballot(pos[s] == position);
               if (b) row = __builtin_ctzll(b) + 64 * s;
            }
            return row;
         };
         auto at_row = [&](int row) {
            T v = lane_value(x[0], row & 63);
            if (S > 1 && row >= 64) v = lane_value(x[S - 1], row & 63);
            return v;
         };
         int p = nelim;
         bool accept = true;
         if (mode == 1) {
            T v;
            p = abs_max(m - 1, v);
            if (p >= m) p = nelim;  // a column without a comparable entry
         } else if (mode == 2) {
            T maxc;
            (void)abs_max(m - 1, maxc);
            p = c;
            if (!(lu_abs(at_row(row_at(c))) >= tu * maxc)) {
               T maxp;
               p = abs_max(k - 1, maxp);
               accept = p < m && lu_abs(at_row(row_at(p))) >= tu * maxc;
            }
         }
         if (accept) {
            prow = row_at(p);
            const T d = T(1) / at_row(prow);
#pragma unroll
            for (int s = 0; s < S; ++s) {
               const int row = lane + 64 * s;
               // below the pivot once the rows at positions nelim and p have changed places
               const bool below = pos[s] >= nelim && row != prow;
               l[s] = x[s] * d;
               if (W > 1) lbuf[par][row] = l[s];
               x[s] = below ? l[s] : x[s];
            }
#pragma unroll
            for (int s = 0; s < S; ++s) {
               if (H == 1 || cc < VL)
                  a[0][s][cc % VL] = x[s];
               else
                  a[H - 1][s][cc % VL] = x[s];
            }
            live &= ~(1u << cc);
         }
         if (W > 1 && lane == 0) ctrl[par] = prow;
      }
      if (W > 1) {
         __syncthreads();
         prow = __builtin_amdgcn_readfirstlane(ctrl[par]);
      }
      if (prow < 0) {  // refused: the next position (mode 2 only)
         ++c;
         continue;
      }
      if (W > 1)
#pragma unroll
         for (int s = 0; s < S; ++s) l[s] = lbuf[par][lane + 64 * s];
      // rows nelim <-> p and columns nelim <-> c change places
      const int plane = prow & 63, ps = prow >> 6;
      int p = lane_value(pos[0], plane);
      if (S > 1 && ps) p = lane_value(pos[S - 1], plane);
#pragma unroll
      for (int s = 0; s < S; ++s) {
         const int row = lane + 64 * s;
         pos[s] = row == prow ? nelim : pos[s] == nelim ? p : pos[s];
      }
      if (mode == 2 && c != nelim && threadIdx.x == 0) {
         colat[c] = colat[nelim];
         colat[nelim] = q;
      }
      auto update = [&](auto sel) {
#pragma unroll
         for (int cidx = 0; cidx < NC; ++cidx) {
            if (!(live >> cidx & 1)) continue;
            const T w = lane_value(a[cidx / VL][sel][cidx % VL], plane);
#pragma unroll
            for (int s = 0; s < S; ++s) {
               const T old = a[cidx / VL][s][cidx % VL];
               a[cidx / VL][s][cidx % VL] = pos[s] > nelim ? fma(-l[s], w, old) : old;
            }
         }
      };
      if (S == 1 || ps == 0)
         update(std::integral_constant<int, 0>{});
      else
         update(std::integral_constant<int, S - 1>{});
      ++nelim;
      c = nelim;
      if (mode == 2 && W > 1) __syncthreads();  // colat
   }
   __syncthreads();
   // column j goes to its position, each row to its own
   for (int j = threadIdx.x; j < m; j += 64 * W) {
      cperm[t.perm + j] = colat[j];
      posof[colat[j]] = j;
   }
   __syncthreads();
#pragma unroll
   for (int c = 0; c < NC; ++c) {
      const int j = c * W + wave;
      if (j >= m) break;
      const int64_t dst = (int64_t)__builtin_amdgcn_readfirstlane(posof[j]) * m;
#pragma unroll
      for (int s = 0; s < S; ++s)
         if (pos[s] >= 0) F[dst + pos[s]] = a[c / VL][s][c % VL];
   }
   if (wave == 0)
#pragma unroll
      for (int s = 0; s < S; ++s)
         if (pos[s] >= 0) rperm[t.perm + pos[s]] = lane + 64 * s;
   if (threadIdx.x == 0) nelim_out[t.front] = nelim;
}

// Fronts by order: one wave up to 32 rows (no barrier), four waves up to 64,
// eight or sixteen with two rows a lane up to 128: the fewest waves whose
// registers hold the front. 20,000 fronts of orders 8 to 128, partial
// pivoting, against the form in LDS: FP64 13.9 -> 3.0 ms, FP32 6.5 -> 1.4 ms
// (threshold pivoting 13.4 -> 3.4, 6.7 -> 1.5 ms).
constexpr int kLuClasses = 3;
inline int lu_class(int m) { return m <= 32 ? 0 : m <= 64 ? 1 : 2; }

template <typename T>
void launch_lu(const LuTask* tasks, const int* count, T* data, int mode, double u, int* rperm, int* cperm, int* nelim,
               hipStream_t s) {
   // FP64: sixteen waves of eight columns (eight waves of sixteen spill in 128 registers)
   constexpr int W2 = sizeof(T) == 8 ? 16 : 8;
   if (count[2] > 0)
      k_lu_front<T, W2, 2, 128 / W2><<<count[2], 64 * W2, 0, s>>>(tasks, data, mode, u, rperm, cperm, nelim);
   tasks += count[2];
   if (count[1] > 0) k_lu_front<T, 4, 1, 16><<<count[1], 256, 0, s>>>(tasks, data, mode, u, rperm, cperm, nelim);
   tasks += count[1];
   if (count[0] > 0) k_lu_front<T, 1, 1, 32><<<count[0], 64, 0, s>>>(tasks, data, mode, u, rperm, cperm, nelim);
}

}  // namespace

int batched_front_lu(int nfronts, const int* m, const int* k, const int64_t* off, void* data, int dtype, int mode,
                     double u, int* rperm, int* cperm, int* nelim, void* stream) {
   if (nfronts < 0 || (nfronts > 0 && (!m || !k || !off || !data || !rperm || !cperm || !nelim)) || mode < 0 ||
       mode > 2 || (dtype != 0 && dtype != 1))
      return SYLVER_ERROR_CALL_SEQUENCE;
   if (nfronts == 0) return 0;
   // the tasks class by class, the largest fronts first
   std::vector<LuTask> tasks(nfronts);
   int count[kLuClasses] = {0, 0, 0}, at[kLuClasses];
   for (int f = 0; f < nfronts; ++f) ++count[lu_class(m[f])];
   at[2] = 0;
   at[1] = count[2];
   at[0] = count[2] + count[1];
   int64_t perm = 0;
   for (int f = 0; f < nfronts; ++f) {
      if (m[f] < 1 || m[f] > kLuMaxRows || k[f] < 0 || k[f] > m[f] || off[f] < 0)
         return SYLVER_ERROR_CALL_SEQUENCE;
      tasks[at[lu_class(m[f])]++] = LuTask{off[f], m[f], k[f], perm, f, 0};
      perm += m[f];
   }
   int dev_count = 0;
   if (hipGetDeviceCount(&dev_count) != hipSuccess || dev_count < 1) return SYLVER_ERROR_CUDA_UNKNOWN;
   hipStream_t s = static_cast<hipStream_t>(stream);
   LuTask* dt = nullptr;
   int *drp = nullptr, *dcp = nullptr, *dne = nullptr;
   int rc = 0;
   auto ok = [&](hipError_t e) {
      if (e != hipSuccess && rc == 0) rc = SYLVER_ERROR_CUDA_UNKNOWN;
      return rc == 0;
   };
   hipEvent_t e0 = nullptr, e1 = nullptr;
   if (ok(hipMalloc(&dt, nfronts * sizeof(LuTask))) && ok(hipMalloc(&drp, perm * sizeof(int))) &&
       ok(hipMalloc(&dcp, perm * sizeof(int))) && ok(hipMalloc(&dne, nfronts * sizeof(int))) &&
       ok(hipEventCreate(&e0)) && ok(hipEventCreate(&e1)) &&
       ok(hipMemcpyAsync(dt, tasks.data(), nfronts * sizeof(LuTask), hipMemcpyHostToDevice, s)) &&
       ok(hipEventRecord(e0, s))) {
      if (dtype == 0)
         launch_lu(dt, count, static_cast<double*>(data), mode, u, drp, dcp, dne, s);
      else
         launch_lu(dt, count, static_cast<float*>(data), mode, u, drp, dcp, dne, s);
      if (ok(hipGetLastError()) && ok(hipEventRecord(e1, s)) &&
          ok(hipMemcpyAsync(rperm, drp, perm * sizeof(int), hipMemcpyDeviceToHost, s)) &&
          ok(hipMemcpyAsync(cperm, dcp, perm * sizeof(int), hipMemcpyDeviceToHost, s)) &&
          ok(hipMemcpyAsync(nelim, dne, nfronts * sizeof(int), hipMemcpyDeviceToHost, s)) &&
          ok(hipStreamSynchronize(s))) {
         float ms = 0;
         if (ok(hipEventElapsedTime(&ms, e0, e1))) set_last_batched_ms(ms);  // the kernel alone
      }
   }
   for (hipEvent_t e : {e0, e1})
      if (e) (void)hipEventDestroy(e);
   for (void* p : {(void*)dt, (void*)drp, (void*)dcp, (void*)dne})
      if (p) (void)hipFree(p);
   return rc;
}

}  // namespace sylver_amd
