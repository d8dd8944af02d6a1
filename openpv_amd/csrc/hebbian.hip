// HebbianUpdater dW for shared weights (HebbianUpdater.cpp:476-627).
//
// EXACT form: one thread per dW element; a wave covers 64 consecutive items
// of one data patch, so the presynaptic activity it walks is wave-uniform.
// For a dW element the reference accumulates (HebbianUpdater.cpp:501-528):
//   batch ascending, then the presynaptic extended rows and columns of that
//   data patch ascending, skipping a_pre == 0, adding (dWMax*a_pre)*a_post.
// Counts (normalizeDw) increment once per contributing presynaptic neuron.
#include "pvhip_internal.hpp"

#include <algorithm>

typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
typedef float f32x8v __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace pvhip {
namespace {

struct HebbParams {
   Geo pre, post;
   int nxp, nyp, nfp;
   int nKx, nKy;
   const int32_t *dimX, *dimY, *pstartX, *pstartY, *apostX, *apostY;
   float dwMax;
   const float *preData, *postData;
   float *dw;
   int64_t *counts;
};

__global__ void __launch_bounds__(256) hebbian_exact_kernel(HebbParams p) {
   int const patchSize  = p.nxp * p.nyp * p.nfp;
   int const numKernels = p.nKx * p.nKy * p.pre.nf;
   size_t const n       = (size_t)numKernels * patchSize;
   size_t const index   = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
   if (index >= n) {
      return;
   }
   int const d    = (int)(index / patchSize);
   int const item = (int)(index % patchSize);
   int const f    = d % p.pre.nf;
   int const dx   = (d / p.pre.nf) % p.nKx;
   int const dy   = d / (p.pre.nf * p.nKx);
   int const F    = item % p.nfp;
   int const wx   = (item / p.nfp) % p.nxp;
   int const wy   = item / (p.nfp * p.nxp);
   int const nxExt = p.pre.nxExt();
   int const nyExt = p.pre.nyExt();
   int const nxExtPost = p.post.nxExt();
   // First extended column/row whose data index is (dx, dy):
   // (xe - lt) mod nKx == dx  (Weights.cpp:212-216).
   int x0 = (dx + p.pre.lt) % p.nKx;
   int y0 = (dy + p.pre.up) % p.nKy;
   float acc   = p.dw[index];
   int64_t cnt = p.counts ? p.counts[index] : 0;
   for (int b = 0; b < p.pre.nbatch; b++) {
      float const *preB  = p.preData + (size_t)b * p.pre.numExt();
      float const *postB = p.postData + (size_t)b * p.post.numExt();
      for (int ye = y0; ye < nyExt; ye += p.nKy) {
         int const ry = wy - p.pstartY[ye];
         bool const rowOk = ry >= 0 && ry < p.dimY[ye];
         for (int xe = x0; xe < nxExt; xe += p.nKx) {
            float const preact = preB[((size_t)ye * nxExt + xe) * p.pre.nf + f];
            if (preact == 0.0f) {
               continue;
            }
            int const rx = wx - p.pstartX[xe];
            if (!rowOk || rx < 0 || rx >= p.dimX[xe]) {
               continue;
            }
            float const apost =
                  postB[((size_t)(p.apostY[ye] + ry) * nxExtPost + p.apostX[xe] + rx) * p.post.nf + F];
            cnt++;
            float t = p.dwMax * preact;
            t       = t * apost;
            acc     = acc + t;
         }
      }
   }
   p.dw[index] = acc;
   if (p.counts) {
      p.counts[index] = cnt;
   }
}

// ------------------------------------------------------------ MFMA correlation
//
// dW[f][item] = dWMax * sum_{b, ye, xe} a_pre[b][ye][xe][f] * P[b](window(ye, xe) + item)
// for connections with one data patch per feature: a GEMM with M = features,
// N = patch items (ky, kx, f'), K = batch x pre extended positions.  P is the
// post activity with every value outside the post restricted region read as
// 0, which is the reference's shrunken patch (pvhost_hebbian_windows checks
// the geometry).
//
// Counts (normalizeDw): an active pre neuron counts for the items of its
// window inside the post restricted region, an interval of window rows times
// an interval of window columns.  Each active neuron is added to the corners of
// its rectangle in an integer difference array D[ky][kx][f], whose
// two-dimensional prefix sums are the counts.  Neurons whose whole window is
// inside, all but a few rows and columns of the layer, add to (0, 0) only: the
// workgroups of the first item block count them as they stage the activity.
// hebbian_border_kernel adds the others.  (Counted by a second correlation, of
// the indicators, they took 710 us beside the 370 us of dW for
// 8 x 128x128x1024 -> 16x16 in BF16, and 96 beside 65 us for
// 7 x 45x37x200 -> 8x8x3 in FP32.)
//
// Workgroup: 64 features x up to 256 items (NB blocks of 16), 4 waves; wave w
// owns features 16w .. 16w+15 for all the items.  K runs over pre extended rows
// (b, ye), 32 columns xe a step.  The A operand (activity) needs no LDS: lane
// (r, g) loads the activity of feature r at columns 8g .. 8g+7, each load a run
// of 16 features per column, HPF steps ahead, and converts it in registers.
// The post rows of the windows are staged in LDS phase-split
// ([ring row][f'][phase][xq], T) so that the values for 8 consecutive pre
// columns xe of one item are 8 consecutive LDS elements; they live in a ring
// (slot = post row mod R), so a pre row following the one before in the same
// image stages only the sy post rows its window advanced by.  With R = nyp + sy
// those are written while the current row is still being read: one barrier a
// row (R = nyp, where the LDS has no room for more, needs two).  A thread's
// elements of a post row are the same for every row, so their offsets are
// computed once.  A lane's 8 K values are pre columns 8g..8g+7 of a step; the
// FP32 form runs eight v_mfma_f32_16x16x4f32, MFMA j taking column 8g+j (the
// same permutation of K for both operands).  BF16 rows are stored twice, the
// second copy shifted by one element, so a fragment starting at any element is
// read as four aligned 32-bit words.
//
// Bound: no single unit; with parts left out in turn, the LDS reads of the
// window fragments, the staging between barriers and the MFMAs cost about a
// fifth each of the large case.  Measured against the form that staged the
// activity through LDS (two barriers and two thousand index instructions a
// row): 8 x 128x128x1024 -> 16x16 BF16 409 -> 277 us, 7 x 45x37x200 -> 8x8x3
// FP32 69 -> 49 us.
constexpr int HMT = 64;  // features per workgroup
constexpr int HNT = 256; // items per workgroup (at most)
constexpr int HPF = 2;   // steps whose activity is in flight
constexpr int HBR = 4;   // post rows and elements per thread prefetched for the next pre row
constexpr int HBI = 3;

struct HebbMfma {
   Geo pre, post;
   int nxp, nyp, nfp, N, nK;
   int sx, cx0, qx0, sy, cy; // window: post ext x = sx*(xq + qx0) + phase, rows sy*ye + cy + ky
   int kxPad, lq, ring;       // 32-padded pre ext width, B row length, ring rows
   int rowsPerChunk;
   const float *preData, *postData;
   float *part; // [chunks][nK][N]
   int *diff;   // [nyp][nxp][nK] differences of the activation counts, or NULL
   int xA, xB, yA, yB; // pre extended columns and rows whose whole window is inside
   float iNfp, iNxp, iSx; // reciprocals of nfp, nxp, sx
};

// n / d by the reciprocal of d, exact for 0 <= n < 2^21 (the items, columns and
// LDS elements of a workgroup): three instructions where an integer division
// by a runtime value takes about forty, and a workgroup's start needs many.
__device__ __forceinline__ int hdiv(int n, float inv) { return (int)(((float)n + 0.5f) * inv); }

template <typename T>
struct HebbFrag;
template <>
struct HebbFrag<__bf16> {
   typedef bf16x8v type;
};
template <>
struct HebbFrag<float> {
   typedef f32x8v type;
};

// B fragment: 8 consecutive elements at p (4-byte aligned).
__device__ __forceinline__ bf16x8v hload_b(const __bf16 *p) {
   const uint32_t *w = reinterpret_cast<const uint32_t *>(p);
   uint32_t v[4] = {w[0], w[1], w[2], w[3]};
   return __builtin_bit_cast(bf16x8v, v);
}
__device__ __forceinline__ f32x8v hload_b(const float *p) {
   f32x8v v;
#pragma unroll
   for (int j = 0; j < 8; j++) {
      v[j] = p[j];
   }
   return v;
}

template <typename T, int NB>
__global__ void __launch_bounds__(256, 2) hebbian_mfma_kernel(HebbMfma h) {
   extern __shared__ float smem[];
   using Frag       = typename HebbFrag<T>::type;
   T *bl            = reinterpret_cast<T *>(smem);
   int const rowB   = h.nfp * h.sx * h.lq;                // B elements of one post row
   int const cstr   = (h.ring * rowB + 7) / 8 * 8;        // elements per B copy (16-byte multiple)
   int const f0     = blockIdx.x * HMT;
   int const n0     = blockIdx.y * HNT;
   int const chunk  = blockIdx.z;
   int const nyExt  = h.pre.nyExt();
   int const nxExt  = h.pre.nxExt();
   int const rows   = h.pre.nbatch * nyExt;
   int const r0     = chunk * h.rowsPerChunk;
   int const r1     = min(r0 + h.rowsPerChunk, rows);
   int const tid    = threadIdx.x;
   int const lane   = tid % 64;
   int const wave   = __builtin_amdgcn_readfirstlane(tid / 64);
   int const r      = lane % 16;
   int const g      = lane / 16;
   int const nxExtP = h.post.nxExt();

   // this lane's item of each item block: window row (upper bits) and the B
   // element offset within a ring row (an odd one in the shifted copy)
   constexpr int KYS = 20; // bits of an LDS element offset
   int item[NB];
#pragma unroll
   for (int nb = 0; nb < NB; nb++) {
      int const n  = min(n0 + nb * 16 + r, h.N - 1);
      int const kp = hdiv(n, h.iNfp); // ky*nxp + kx
      int const fp = n - kp * h.nfp;
      int const ky = hdiv(kp, h.iNxp);
      int const px = h.cx0 + kp - ky * h.nxp;
      int const xq = hdiv(px, h.iSx);
      int sub      = (fp * h.sx + px - xq * h.sx) * h.lq + xq + 8 * g;
      if (sizeof(T) == 2 && (sub & 1)) { // lq and x0 are even: the parity stays
         sub += cstr - 1;
      }
      item[nb] = ky << KYS | sub;
   }
   f32x4 acc[NB];
#pragma unroll
   for (int nb = 0; nb < NB; nb++) {
      acc[nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
   }

   // ---- post rows -> LDS.  Element i of a post row is post column i / nfp of
   // the staged range, feature i % nfp.
   int const bItems = h.sx * h.lq * h.nfp;
   auto b_item = [&](int i, int &loff, int &goff) {
      int const pxr = hdiv(i, h.iNfp);
      int const c   = i - pxr * h.nfp;
      int const px  = pxr + h.sx * h.qx0;
      int const xq  = hdiv(pxr, h.iSx);
      loff          = (c * h.sx + pxr - xq * h.sx) * h.lq + xq;
      goff          = px >= h.post.lt && px < h.post.lt + h.post.nx ? px * h.nfp + c : -1;
   };
   int bL[HBI], bG[HBI]; // offsets of this thread's first HBI elements
#pragma unroll
   for (int u = 0; u < HBI; u++) {
      int const i = tid + 256 * u;
      b_item(min(i, bItems - 1), bL[u], bG[u]);
      bL[u] = i < bItems ? bL[u] : -1;
   }
   auto slot_of = [&](int py) {
      int const m = py % h.ring;
      return m < 0 ? m + h.ring : m;
   };
   auto wrap = [&](int slot) {
      while (slot >= h.ring) {
         slot -= h.ring;
      }
      return slot;
   };
   // post row py of batch element b, or NULL outside the restricted rows
   auto post_row = [&](int b, int py) -> const float * {
      return py >= h.post.up && py < h.post.up + h.post.ny
                   ? h.postData + (size_t)b * h.post.numExt() + (size_t)py * nxExtP * h.nfp
                   : nullptr;
   };
   auto b_get = [&](const float *P, int goff) { return P && goff >= 0 ? P[goff] : 0.0f; };
   auto b_put = [&](int slot, int loff, float v) {
      int const idx = slot * rowB + loff;
      T const x     = (T)v;
      bl[idx]       = x;
      if (sizeof(T) == 2 && idx > 0) {
         bl[cstr + idx - 1] = x; // copy 1: shifted left by one element
      }
   };
   auto stage_rest = [&](const float *P, int slot) __attribute__((always_inline)) { // elements past the prefetched ones
      for (int i = tid + 256 * HBI; i < bItems; i += 256) {
         int lo, go;
         b_item(i, lo, go);
         b_put(slot, lo, b_get(P, go));
      }
   };
   // n post rows from py: the first HBR of them into registers, then to LDS
   float vb[HBR][HBI];
   auto fetch_rows = [&](int b, int py, int n) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < HBR; j++) {
         const float *P = j < n ? post_row(b, py + j) : nullptr;
#pragma unroll
         for (int u = 0; u < HBI; u++) {
            vb[j][u] = bL[u] >= 0 ? b_get(P, bG[u]) : 0.0f;
         }
      }
   };
   // (slot: ring row of post row py)
   auto put_rows = [&](int b, int py, int slot, int n) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < HBR; j++) {
         if (j < n) {
#pragma unroll
            for (int u = 0; u < HBI; u++) {
               if (bL[u] >= 0) {
                  b_put(slot, bL[u], vb[j][u]);
               }
            }
            stage_rest(post_row(b, py + j), slot);
            slot = slot + 1 < h.ring ? slot + 1 : 0;
         }
      }
   };
   auto stage_rows = [&](int b, int py, int slot, int n) __attribute__((always_inline)) {
      for (int j = 0; j < n; j += HBR) {
         fetch_rows(b, py + j, n - j);
         put_rows(b, py + j, wrap(slot + j), n - j);
      }
   };
   // The current pre row: batch element, row, its window's first post row and
   // that row's ring slot.  The next row of the image continues its window: sy
   // new post rows.
   int cb = r0 / nyExt, ye = r0 - cb * nyExt;
   int wy = h.sy * ye + h.cy, slot0 = slot_of(wy);
   auto continues = [&]() { return ye + 1 < nyExt && h.sy < h.nyp; };
   auto fetch_new = [&]() __attribute__((always_inline)) { fetch_rows(cb, wy + h.nyp, h.sy); };
   auto stage_new = [&]() __attribute__((always_inline)) { // before the step to that row
      put_rows(cb, wy + h.nyp, wrap(slot0 + h.nyp), h.sy);
      stage_rows(cb, wy + h.nyp + HBR, wrap(slot0 + h.nyp + HBR), h.sy - HBR);
   };
   auto stage_window = [&]() __attribute__((always_inline)) { stage_rows(cb, wy, slot0, h.nyp); };
   auto next_row = [&]() {
      if (++ye < nyExt) {
         wy += h.sy;
         slot0 = wrap(slot0 + h.sy);
      }
      else {
         ye = 0;
         cb++;
         wy    = h.cy;
         slot0 = slot_of(wy);
      }
   };

   // ---- activity: step q of the chunk is row r0 + q / steps, columns
   // 32*(q % steps) ..; the loads of step q + HPF are issued in step q
   int const steps  = h.kxPad / 32;
   int const nSteps = (r1 - r0) * steps;
   int const f      = min(f0 + wave * 16 + r, h.nK - 1); // rows past the last feature are not stored
   float va[HPF][8];
   int lRow = r0, lX = 0; // of the next load
   uint32_t aoff[8];      // element of column 8g + j of a step
#pragma unroll
   for (int j = 0; j < 8; j++) {
      aoff[j] = (uint32_t)((8 * g + j) * h.nK + f);
   }
   auto load_a = [&](float (&v)[8]) __attribute__((always_inline)) {
      float const *base = h.preData + ((size_t)lRow * nxExt + lX) * h.nK;
      if (lX + 32 <= nxExt) {
#pragma unroll
         for (int j = 0; j < 8; j++) {
            v[j] = base[aoff[j]];
         }
      }
      else { // columns past the layer read its last one and are cleared before use
#pragma unroll
         for (int j = 0; j < 8; j++) {
            v[j] = base[(uint32_t)(min(8 * g + j, nxExt - 1 - lX) * h.nK + f)];
         }
      }
      lX += 32;
      if (lX >= h.kxPad) {
         lX   = 0;
         lRow = min(lRow + 1, r1 - 1); // past the end: loaded, not used
      }
   };
   bool const counting = h.diff != nullptr && blockIdx.y == 0 && f0 + wave * 16 + r < h.nK;
   int active          = 0; // active neurons of feature f with a whole window
   if (r0 < r1) {
#pragma unroll
      for (int s = 0; s < HPF; s++) {
         load_a(va[s]);
      }
      stage_window();
   }
   __syncthreads();
   int row = r0, x0 = 0;
   int bb[NB]; // B element of this row's fragments at column 0
   auto bases = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
         int s  = slot0 + (item[nb] >> KYS);
         s      = s >= h.ring ? s - h.ring : s;
         bb[nb] = s * rowB + (item[nb] & ((1 << KYS) - 1));
      }
   };
   if (r0 < r1) {
      bases();
   }
   for (int q0 = 0; q0 < nSteps; q0 += HPF) {
#pragma unroll
      for (int s = 0; s < HPF; s++) {
         if (q0 + s < nSteps) { // the same for the whole workgroup
            if (x0 == 0 && row + 1 < r1 && continues()) {
               fetch_new(); // in flight during this row
            }
            bool const tail = x0 + 32 > nxExt;
            if (tail) { // columns past the layer
#pragma unroll
               for (int j = 0; j < 8; j++) {
                  va[s][j] = x0 + 8 * g + j < nxExt ? va[s][j] : 0.0f;
               }
            }
            if (counting && ye >= h.yA && ye < h.yB) {
               if (x0 >= h.xA && x0 + 32 <= h.xB) {
#pragma unroll
                  for (int j = 0; j < 8; j++) {
                     active += va[s][j] != 0.0f ? 1 : 0;
                  }
               }
               else {
#pragma unroll
                  for (int j = 0; j < 8; j++) {
                     int const xe = x0 + 8 * g + j;
                     active += va[s][j] != 0.0f && xe >= h.xA && xe < h.xB ? 1 : 0;
                  }
               }
            }
            Frag af;
#pragma unroll
            for (int j = 0; j < 8; j++) {
               af[j] = (T)va[s][j];
            }
            load_a(va[s]); // step q0 + s + HPF
            // B fragments a group ahead of their MFMAs
            constexpr int G = sizeof(T) == 2 ? 4 : 1;
            Frag bf[2][G];
#pragma unroll
            for (int k = 0; k < G; k++) {
               bf[0][k] = hload_b(bl + bb[k] + x0);
            }
#pragma unroll
            for (int nb = 0; nb < NB; nb += G) {
#pragma unroll
               for (int k = 0; k < G; k++) {
                  if (nb + G < NB) {
                     bf[(nb / G + 1) % 2][k] = hload_b(bl + bb[(nb + G) % NB + k] + x0);
                  }
               }
               __builtin_amdgcn_sched_barrier(0);
#pragma unroll
               for (int k = 0; k < G; k++) {
                  Frag const b = bf[nb / G % 2][k];
                  if constexpr (sizeof(T) == 2) {
                     acc[nb + k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, b, acc[nb + k], 0, 0, 0);
                  }
                  else {
#pragma unroll
                     for (int j = 0; j < 8; j++) {
                        acc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[j], b[j], acc[nb], 0, 0, 0);
                     }
                  }
               }
            }
            x0 += 32;
            if (x0 >= h.kxPad) { // the next row
               x0 = 0;
               if (row + 1 < r1) {
                  bool const next = continues();
                  if (!next || h.ring == h.nyp) {
                     __syncthreads(); // this row's fragments are consumed
                  }
                  row++;
                  if (next) {
                     stage_new();
                  }
                  next_row();
                  if (!next) {
                     stage_window();
                  }
                  __syncthreads();
                  bases();
               }
            }
         }
      }
   }
   if (counting && active > 0) {
      atomicAdd(h.diff + f, active);
   }
   // D[4g+i][r]: feature f0 + 16*wave + 4g + i, item of lane r in block nb
   float *out = h.part + (size_t)chunk * h.nK * h.N;
#pragma unroll
   for (int nb = 0; nb < NB; nb++) {
      int const n = n0 + nb * 16 + r;
#pragma unroll
      for (int i = 0; i < 4; i++) {
         int const fo = f0 + wave * 16 + 4 * g + i;
         if (fo < h.nK && n < h.N) {
            out[(size_t)fo * h.N + n] = acc[nb][i];
         }
      }
   }
}

// Counts of the pre neurons whose window is cut by the edge of the post
// restricted region: one thread per feature and segment of up to kBorderRun
// neurons with the same rectangle -- a run of whole rows of a cut column, a run
// of whole columns of a cut row, or one neuron where both are cut.
constexpr int kBorderRun = 32;

__global__ void __launch_bounds__(256) hebbian_border_kernel(HebbMfma h) {
   int const f     = blockIdx.y * kWave + threadIdx.x % kWave;
   int seg         = blockIdx.x * (256 / kWave) + threadIdx.x / kWave;
   int const nxExt = h.pre.nxExt();
   int const nyExt = h.pre.nyExt();
   int const nbx   = nxExt - (h.xB - h.xA); // cut columns, rows
   int const nby   = nyExt - (h.yB - h.yA);
   int const runsY = (h.yB - h.yA + kBorderRun - 1) / kBorderRun;
   int const runsX = (h.xB - h.xA + kBorderRun - 1) / kBorderRun;
   int const per   = nbx * runsY + nby * runsX + nby * nbx; // segments of a batch element
   int const b     = seg / per;
   if (b >= h.pre.nbatch || f >= h.nK) {
      return;
   }
   seg -= b * per;
   auto cut_x = [&](int i) { return i < h.xA ? i : i - h.xA + h.xB; };
   auto cut_y = [&](int i) { return i < h.yA ? i : i - h.yA + h.yB; };
   int xe, ye, n, step = 0; // first neuron, their number, positions from one to the next
   if (seg < nbx * runsY) {
      xe   = cut_x(seg / runsY);
      ye   = h.yA + seg % runsY * kBorderRun;
      n    = min(kBorderRun, h.yB - ye);
      step = nxExt;
   }
   else if (seg < nbx * runsY + nby * runsX) {
      seg -= nbx * runsY;
      ye   = cut_y(seg / runsX);
      xe   = h.xA + seg % runsX * kBorderRun;
      n    = min(kBorderRun, h.xB - xe);
      step = 1;
   }
   else {
      seg -= nbx * runsY + nby * runsX;
      ye = cut_y(seg / nbx);
      xe = cut_x(seg % nbx);
      n  = 1;
   }
   // rectangle [ya, yb) x [xa, xb) of window items inside the restricted region
   int const sx = h.sx * (xe + h.qx0) + h.cx0;
   int const sy = h.sy * ye + h.cy;
   int const xa = max(0, min(h.nxp, h.post.lt - sx));
   int const xb = max(0, min(h.nxp, h.post.lt + h.post.nx - sx));
   int const ya = max(0, min(h.nyp, h.post.up - sy));
   int const yb = max(0, min(h.nyp, h.post.up + h.post.ny - sy));
   if (xa >= xb || ya >= yb) {
      return;
   }
   float const *v = h.preData + (((size_t)b * nyExt + ye) * nxExt + xe) * h.nK + f;
   int on         = 0;
#pragma unroll 8
   for (int i = 0; i < n; i++) {
      on += v[(size_t)i * step * h.nK] != 0.0f ? 1 : 0;
   }
   if (on > 0) {
      atomicAdd(h.diff + (ya * h.nxp + xa) * h.nK + f, on);
      if (xb < h.nxp) {
         atomicAdd(h.diff + (ya * h.nxp + xb) * h.nK + f, -on);
      }
      if (yb < h.nyp) {
         atomicAdd(h.diff + (yb * h.nxp + xa) * h.nK + f, -on);
         if (xb < h.nxp) {
            atomicAdd(h.diff + (yb * h.nxp + xb) * h.nK + f, on);
         }
      }
   }
}

// dw[f][n] += dWMax * sum_c part[c][f][n] (chunks in order, eight loads in
// flight); counts[f][n] += the prefix sum of diff[..][..][f] at the item's
// window row and column.  Grid (features, ceil(N / 256)).
__global__ void __launch_bounds__(256) hebbian_reduce_kernel(
      const float *part, const int *diff, int chunks, int N, int nyp, int nxp, int nfp, float dwMax, float *dw,
      int64_t *counts) {
   extern __shared__ int sums[]; // [nyp][nxp]
   int const f    = blockIdx.x;
   int const tid  = threadIdx.x;
   if (counts) {
      int const items = nyp * nxp;
      for (int i = tid; i < items; i += 256) {
         sums[i] = diff[(size_t)i * gridDim.x + f];
      }
      __syncthreads();
      for (int y = tid; y < nyp; y += 256) {
         for (int x = 1; x < nxp; x++) {
            sums[y * nxp + x] += sums[y * nxp + x - 1];
         }
      }
      __syncthreads();
      for (int x = tid; x < nxp; x += 256) {
         for (int y = 1; y < nyp; y++) {
            sums[y * nxp + x] += sums[(y - 1) * nxp + x];
         }
      }
      __syncthreads();
   }
   int const n = blockIdx.y * 256 + tid;
   if (n >= N) {
      return;
   }
   size_t const i      = (size_t)f * N + n;
   size_t const stride = (size_t)gridDim.x * N;
   float s             = 0.0f;
   int c               = 0;
   for (; c + 8 <= chunks; c += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
         v[u] = part[(size_t)(c + u) * stride + i];
      }
#pragma unroll
      for (int u = 0; u < 8; u++) {
         s = s + v[u];
      }
   }
   for (; c < chunks; c++) {
      s = s + part[(size_t)c * stride + i];
   }
   dw[i] = dw[i] + dwMax * s;
   if (counts) {
      counts[i] += sums[n / nfp];
   }
}

struct HebbPlan {
   int chunks, rowsPerChunk, kxPad, lq, ring;
   size_t lds, partBytes;
   size_t diffBytes; // difference array of the counts
};

HebbPlan hebb_plan(const pvhip_hebbian_args &a, bool bf) {
   HebbPlan pl;
   Geo pre    = geo(a.pre);
   int nK     = a.pre.nf;
   int N      = a.nxp * a.nyp * a.nfp;
   int mt     = (nK + HMT - 1) / HMT;
   int nt     = (N + HNT - 1) / HNT;
   int rows   = pre.nbatch * pre.nyExt();
   // enough workgroups to fill the chip twice, at least 4 rows per chunk
   // (or the caller's choice)
   int want   = std::max(1, 512 / std::max(1, mt * nt));
   pl.rowsPerChunk = a.rows_per_chunk > 0 ? std::min(a.rows_per_chunk, rows)
                                          : std::max(4, (rows + want - 1) / want);
   pl.chunks       = (rows + pl.rowsPerChunk - 1) / pl.rowsPerChunk;
   pl.kxPad        = (pre.nxExt() + 31) / 32 * 32;
   int sx          = std::max(1, a.window_stride_x);
   int cx          = a.window_start_x;
   int qx0         = cx >= 0 ? cx / sx : -((-cx + sx - 1) / sx);
   int cx0         = cx - sx * qx0;
   pl.lq           = (pl.kxPad + (cx0 + a.nxp - 1) / sx + 2 + 1) / 2 * 2;
   size_t esz      = bf ? 2 : 4;
   int copies      = bf ? 2 : 1;
   auto lds_of     = [&](int ring) {
      return copies * (((size_t)ring * a.nfp * sx * pl.lq + 7) / 8 * 8) * esz;
   };
   // room for the rows of the next window beside the current one's, unless
   // that leaves one workgroup per CU
   pl.ring = a.nyp + std::max(1, a.window_stride_y);
   if (lds_of(pl.ring) > 80 * 1024) {
      pl.ring = a.nyp;
   }
   pl.lds = lds_of(pl.ring);
   pl.partBytes    = (size_t)pl.chunks * nK * N * sizeof(float);
   pl.diffBytes    = a.counts ? (size_t)nK * a.nyp * a.nxp * sizeof(int) : 0;
   return pl;
}

} // namespace
} // namespace pvhip

using namespace pvhip;

extern "C" {

int pvhip_hebbian_dw(const pvhip_hebbian_args *a, pvhip_stream stream) {
   PVHIP_REQUIRE(a != nullptr, "pvhip_hebbian_dw: NULL args");
   PVHIP_REQUIRE(loc_valid(a->pre) && loc_valid(a->post), "hebbian_dw: invalid loc");
   PVHIP_REQUIRE(a->pre.nbatch == a->post.nbatch, "hebbian_dw: batch sizes differ");
   PVHIP_REQUIRE(a->nfp == a->post.nf, "hebbian_dw: nfp must equal post nf");
   PVHIP_REQUIRE(a->num_kernels_x > 0 && a->num_kernels_y > 0, "hebbian_dw: bad kernel counts");
   PVHIP_REQUIRE(
         a->dim_x && a->dim_y && a->pstart_x && a->pstart_y && a->apost_x && a->apost_y,
         "hebbian_dw: NULL geometry table");
   PVHIP_REQUIRE(a->pre_data && a->post_data && a->dw, "hebbian_dw: NULL buffer");
   PVHIP_REQUIRE(a->rows_per_chunk >= 0, "hebbian_dw: negative rows_per_chunk");
   if (a->arith == PVHIP_ARITH_FP32 || a->arith == PVHIP_ARITH_BF16) {
      bool const bf = a->arith == PVHIP_ARITH_BF16;
      PVHIP_REQUIRE(a->num_kernels_x == 1 && a->num_kernels_y == 1,
            "hebbian_dw: the MFMA forms need one data patch per feature");
      PVHIP_REQUIRE(a->window_stride_x > 0 && a->window_stride_y > 0,
            "hebbian_dw: the MFMA forms need the window geometry (pvhost_hebbian_windows)");
      HebbPlan pl = hebb_plan(*a, bf);
      size_t need = pl.partBytes + pl.diffBytes;
      PVHIP_REQUIRE(a->scratch && a->scratch_bytes >= need,
            "hebbian_dw: scratch of %zu bytes, %zu needed", a->scratch_bytes, need);
      PVHIP_REQUIRE(pl.lds <= 160 * 1024, "hebbian_dw: tile needs %zu bytes of LDS", pl.lds);
      HebbMfma h{};
      h.pre     = geo(a->pre);
      h.post    = geo(a->post);
      h.nxp     = a->nxp;
      h.nyp     = a->nyp;
      h.nfp     = a->nfp;
      h.N       = a->nxp * a->nyp * a->nfp;
      h.nK      = a->pre.nf;
      h.sx      = a->window_stride_x;
      h.qx0     = a->window_start_x >= 0 ? a->window_start_x / h.sx
                                         : -((-a->window_start_x + h.sx - 1) / h.sx);
      h.cx0     = a->window_start_x - h.sx * h.qx0;
      h.sy      = a->window_stride_y;
      h.cy      = a->window_start_y;
      h.kxPad   = pl.kxPad;
      h.lq      = pl.lq;
      h.ring    = pl.ring;
      h.iNfp    = 1.0f / (float)h.nfp;
      h.iNxp    = 1.0f / (float)h.nxp;
      h.iSx     = 1.0f / (float)h.sx;
      h.rowsPerChunk = pl.rowsPerChunk;
      h.preData  = a->pre_data;
      h.postData = a->post_data;
      float *part  = static_cast<float *>(a->scratch);
      dim3 grid((h.nK + HMT - 1) / HMT, (h.N + HNT - 1) / HNT, pl.chunks);
      hipStream_t s = (hipStream_t)stream;
      h.part        = part;
      h.diff        = a->counts ? reinterpret_cast<int *>(part + pl.partBytes / sizeof(float)) : nullptr;
      if (h.diff) {
         int st = pvhip_fill_zero(h.diff, pl.diffBytes, stream);
         if (st) {
            return st;
         }
         // whole windows: start >= lo and start + patch <= lo + n
         auto whole = [](int start0, int stride, int lo, int n, int patch, int ext, int &first, int &end) {
            int const a = lo - start0, z = lo + n - patch - start0;
            first       = std::min(ext, a > 0 ? (a + stride - 1) / stride : 0);
            end         = z < 0 ? 0 : std::min(ext, z / stride + 1);
            if (end <= first) {
               first = end = 0;
            }
         };
         whole(a->window_start_x, h.sx, h.post.lt, h.post.nx, h.nxp, h.pre.nxExt(), h.xA, h.xB);
         whole(a->window_start_y, h.sy, h.post.up, h.post.ny, h.nyp, h.pre.nyExt(), h.yA, h.yB);
      }
      // item blocks of 16 a workgroup holds accumulators for
      int const nb = (std::min(h.N, HNT) + 15) / 16;
#define PVHIP_HEBB(NBV)                                                                                  \
   do {                                                                                                 \
      if (bf) {                                                                                         \
         hipLaunchKernelGGL((hebbian_mfma_kernel<__bf16, NBV>), grid, dim3(256), pl.lds, s, h);          \
      }                                                                                                 \
      else {                                                                                            \
         hipLaunchKernelGGL((hebbian_mfma_kernel<float, NBV>), grid, dim3(256), pl.lds, s, h);           \
      }                                                                                                 \
   } while (0)
      if (nb <= 4) PVHIP_HEBB(4);
      else if (nb <= 8) PVHIP_HEBB(8);
      else if (nb <= 12) PVHIP_HEBB(12);
      else PVHIP_HEBB(16);
#undef PVHIP_HEBB
      PVHIP_LAUNCHED("hebbian_mfma");
      if (h.diff) {
         long long const nbx = h.pre.nxExt() - (h.xB - h.xA), nby = h.pre.nyExt() - (h.yB - h.yA);
         long long const segs = (nbx * ((h.yB - h.yA + kBorderRun - 1) / kBorderRun)
                                 + nby * ((h.xB - h.xA + kBorderRun - 1) / kBorderRun) + nby * nbx)
                                * h.pre.nbatch;
         if (segs > 0) {
            hipLaunchKernelGGL(hebbian_border_kernel, dim3((unsigned)((segs + 3) / 4), (h.nK + kWave - 1) / kWave),
                  dim3(256), 0, s, h);
            PVHIP_LAUNCHED("hebbian_border");
         }
      }
      hipLaunchKernelGGL(hebbian_reduce_kernel, dim3(h.nK, (h.N + 255) / 256), dim3(256),
            a->counts ? (size_t)a->nyp * a->nxp * sizeof(int) : 0, s, part, h.diff, pl.chunks, h.N, a->nyp, a->nxp,
            a->nfp, a->dw_max, a->dw, a->counts);
      PVHIP_LAUNCHED("hebbian_reduce");
      return PVHIP_OK;
   }
   if (a->arith != PVHIP_ARITH_EXACT) {
      return set_error(PVHIP_ERR_UNSUPPORTED, "hebbian_dw: arith %d not built", a->arith);
   }
   HebbParams p;
   p.pre      = geo(a->pre);
   p.post     = geo(a->post);
   p.nxp      = a->nxp;
   p.nyp      = a->nyp;
   p.nfp      = a->nfp;
   p.nKx      = a->num_kernels_x;
   p.nKy      = a->num_kernels_y;
   p.dimX     = a->dim_x;
   p.dimY     = a->dim_y;
   p.pstartX  = a->pstart_x;
   p.pstartY  = a->pstart_y;
   p.apostX   = a->apost_x;
   p.apostY   = a->apost_y;
   p.dwMax    = a->dw_max;
   p.preData  = a->pre_data;
   p.postData = a->post_data;
   p.dw       = a->dw;
   p.counts   = a->counts;
   size_t n   = (size_t)p.nKx * p.nKy * p.pre.nf * p.nxp * p.nyp * p.nfp;
   hipLaunchKernelGGL(hebbian_exact_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
         (hipStream_t)stream, p);
   PVHIP_LAUNCHED("hebbian_exact");
   return PVHIP_OK;
}

size_t pvhip_hebbian_dw_scratch_bytes(const pvhip_hebbian_args *a) {
   if (!a || !loc_valid(a->pre) || a->window_stride_x <= 0 || a->nxp <= 0 || a->nyp <= 0 || a->nfp <= 0) {
      return 0;
   }
   HebbPlan pl = hebb_plan(*a, a->arith == PVHIP_ARITH_BF16);
   return pl.partBytes + pl.diffBytes;
}

} // extern "C"
