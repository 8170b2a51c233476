// bf16 GEMM of prefill-size forwards: Y = X . W^T for more rows than one
// verify round has (vnx_gemm_bf16 / vnx_gemm_bf16_residual past kWgMinM rows),
// and the routed MoD expert products of such forwards
// (vnx_expert_gemm_bf16_rows; mod.py:466-600 evaluated on each expert's own
// rows).  W comes in the packed operand order of gemm.hip (one contiguous KB
// per wave load), so only X goes through LDS.
//
// A workgroup owns RT 32-row tiles of X and 4 CT 32-column tiles of W: wave w
// takes columns (4 gi + w) CT .. + CT and all rows, so a W operand is loaded by
// one wave only (straight to registers, reused over RT row tiles) and an X
// operand read from LDS feeds CT products.  X is double-buffered, one barrier
// per 64-k chunk: chunk c + 1 goes to LDS and a later one to registers while
// chunk c is multiplied.
//
// What bounds it: the matrix cores, less the waits that too few waves leave
// open (loading no W at all, the MoD gate-up below would run at 1.6 PFLOP/s).
// Two things decided the shapes.  Left alone, the compiler sinks every load to
// the end of a chunk and then waits for all of them, so scheduling barriers
// pin each load where it is written; and registers spent on a deeper ring or
// on all A operands at once cost a resident workgroup, which costs more than
// they gain.  MoD gate-up of 2,048 rows (16 experts of 5,376 x 1,024, half of
// the rows each): 196 us, 919 TFLOP/s; down product 108 us, 833 TFLOP/s (the
// dense batched library products they replace: 505 us for both, every expert
// on every row).
#include <climits>

#include "gemm_tiles.h"

namespace vnx {
namespace {

constexpr int kWgNtW = 1, kWgNtY = 2;

// 16 bytes of W; NT: past the caches.
template <bool NT>
__device__ __forceinline__ u32x4 ld_w(const uint16_t* p) {
  if constexpr (NT) return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  else return *reinterpret_cast<const u32x4*>(p);
}

// RT x CT tiles per wave; PD register sets of W and X (PD 1: one set, each W
// register reloaded as soon as its products are issued); LA: A operands of LA
// 16-k steps read ahead (PD 1; else the whole chunk's); OCC workgroups per CU; CP:
// W is read (kWgNtW) or the outputs are written (kWgNtY) past the caches
// (wg_run's rules).
template <int OT, int EPI, int RT, int CT, int PD, int LA, int OCC, int CP = 0>
__global__ __launch_bounds__(256, OCC) void k_wgemm(WgParams p) {
  constexpr bool NT = CP & kWgNtW, NTY = CP & kWgNtY;
  constexpr int ROWS = 32 * RT;
  constexpr int UN = PD;
  constexpr int SLAB = ROWS * kVgRowB;
  constexpr int TP = 36;                       // row pitch (floats) of the output transpose tiles
  constexpr int SM = 2 * SLAB > 4 * 32 * TP * 4 ? 2 * SLAB : 4 * 32 * TP * 4;
  __shared__ __attribute__((aligned(16))) char smem[SM];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // The live tiles, numbered by (group, N group, row tile), are cut into eight
  // equal runs, one per XCD (workgroup t on XCD t % 8): the row tiles that
  // share a group's W columns, and the N groups that share its rows, follow
  // each other on one XCD, and every XCD has the same number of tiles however
  // the rows are routed.
  int z = 0, gi, mi, cnt = p.M;
  {
    int total = 0;
    if (p.counts) {
      for (int e = 0; e < p.batch; ++e) total += (max(min(p.counts[e], p.M), 0) + ROWS - 1) / ROWS;
    } else {
      total = p.batch * ((p.M + ROWS - 1) / ROWS);
    }
    total *= p.ng;
    const int run = (total + kVgXcds - 1) / kVgXcds, at = blockIdx.x >> 3;
    int idx = (blockIdx.x & 7) * run + at;
    if (at >= run || idx >= total) return;     // uniform over the workgroup
    int mt = (p.M + ROWS - 1) / ROWS;
    if (p.counts) {
      for (;; ++z) {
        cnt = max(min(p.counts[z], p.M), 0);
        mt = (cnt + ROWS - 1) / ROWS;
        if (idx < mt * p.ng) break;
        idx -= mt * p.ng;
      }
    } else {
      z = idx / (mt * p.ng);
      idx -= z * mt * p.ng;
    }
    gi = idx / mt;
    mi = idx - gi * mt;
  }
  const int m0 = mi * ROWS;
  const int r = lane & 31, h = lane >> 5;
  const int nch = p.K / kVgChunk;

  // staging: thread tid takes rows tid / 8 + 32 q, 16-byte column tid % 8;
  // rows past the count re-read the last one (computed, never stored)
  const int xr = tid >> 3, xc = tid & 7;
  const uint16_t* xp[RT];
#pragma unroll
  for (int q = 0; q < RT; ++q) {
    const int j = min(m0 + xr + 32 * q, cnt - 1);
    const int64_t row = p.rows ? p.rows[(int64_t)z * p.M + j] : j;
    xp[q] = p.x + z * p.sxb + row * p.ldx + xc * 8;
  }
  const uint16_t* wt[CT];
  int ni[CT];
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    ni[t] = (gi * 4 + wave) * CT + t;          // past nt: computes, never stores
    wt[t] = p.w + z * p.swb + (int64_t)min(ni[t], p.nt - 1) * nch * 2048 + lane * 8;
  }

  f32x16 acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][t][e] = 0.0f;

  // chunk c lives in register set c % PD of W and of X
  u32x4 xv[PD][RT], wv[PD][CT][4];
  auto load_x = [&](int c, u32x4 (&v)[RT]) {
    c = min(c, nch - 1);
#pragma unroll
    for (int q = 0; q < RT; ++q) v[q] = *reinterpret_cast<const u32x4*>(xp[q] + c * kVgChunk);
  };
  auto stage_x = [&](int c, const u32x4 (&v)[RT]) {
    char* buf = smem + (c & 1) * SLAB;
#pragma unroll
    for (int q = 0; q < RT; ++q) *reinterpret_cast<u32x4*>(buf + xs_off(xr + 32 * q, xc)) = v[q];
  };
  auto load_w = [&](int c, u32x4 (&v)[CT][4]) {
    const int64_t cc = min(c, nch - 1);
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int s = 0; s < 4; ++s) v[t][s] = ld_w<NT>(wt[t] + (cc * 4 + s) * 512);
  };
  // Every load in the order of the loop, X(c + 1) before W(c): the waits the
  // compiler derives for the loop's first chunk then leave as many loads in
  // flight as those of a later one.
  load_x(0, xv[0]);
  stage_x(0, xv[0]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int d = 0; d < PD; ++d) {
    load_x(d + 1, xv[(d + 1) % PD]);
    __builtin_amdgcn_sched_barrier(0);
    load_w(d, wv[d]);
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
  for (int c0 = 0; c0 < nch; c0 += UN) {
#pragma unroll
    for (int d = 0; d < UN; ++d) {
      const int c = c0 + d;
      const char* xb = smem + (c & 1) * SLAB;
      constexpr int NA = PD == 1 ? LA : 4;
      u32x4 a[4][RT];
#pragma unroll
      for (int s = 0; s < NA; ++s)
#pragma unroll
        for (int i = 0; i < RT; ++i)
          a[s][i] = *reinterpret_cast<const u32x4*>(xb + xs_off(i * 32 + r, h * 4 + s));
      __builtin_amdgcn_sched_barrier(0);
      stage_x(c + 1, xv[(d + 1) % PD]);        // past the end: the last chunk again, never read
      load_x(c + 1 + PD, xv[(d + 1) % PD]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (PD == 1) {
        const int64_t cw = min(c + 1, nch - 1);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          if (s + NA < 4)
#pragma unroll
            for (int i = 0; i < RT; ++i)
              a[s + NA][i] = *reinterpret_cast<const u32x4*>(xb + xs_off(i * 32 + r, h * 4 + s + NA));
#pragma unroll
          for (int t = 0; t < CT; ++t)
#pragma unroll
            for (int i = 0; i < RT; ++i)
              acc[i][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_b8(a[s][i]), as_b8(wv[0][t][s]), acc[i][t], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int t = 0; t < CT; ++t) wv[0][t][s] = ld_w<NT>(wt[t] + (cw * 4 + s) * 512);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        if (c < nch) {                         // uniform
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int t = 0; t < CT; ++t)
#pragma unroll
              for (int i = 0; i < RT; ++i)
                acc[i][t] =
                    __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_b8(a[s][i]), as_b8(wv[d][t][s]), acc[i][t], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_w(c + PD, wv[d]);
      }
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
    }
  }

  // Each 32 x 32 tile leaves through this wave's LDS tile: lane (r, h) writes
  // D[8ii + 4h + e][r], then lane l holds row l / 2's columns 16 (l % 2) .. +16
  // and stores them as 16- or 32-byte pieces.
  char* ybase = static_cast<char*>(p.y) + (int64_t)z * p.syb * (OT == 0 ? 4 : 2);
  float* tr = reinterpret_cast<float*>(smem) + wave * 32 * TP;
  const int hf = lane & 1;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int j = m0 + i * 32 + (lane >> 1);
    if (m0 + i * 32 >= cnt) continue;          // uniform
    const bool live = j < cnt;
    float cw = 1.0f;
    if (EPI == 1 && p.comb && live)
      cw = p.comb[(p.rows ? p.rows[(int64_t)z * p.M + j] : (int64_t)j) * p.ldc + z];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      if (ni[t] >= p.nt) continue;             // uniform per wave
      if (p.vec_out) {
        f32x4 old[EPI == 3 ? 4 : 1];
        float* yf = reinterpret_cast<float*>(ybase) + (int64_t)j * p.ldy + ni[t] * 32 + 16 * hf;
        if constexpr (EPI == 3) {
          if (live)
#pragma unroll
            for (int q = 0; q < 4; ++q) old[q] = *reinterpret_cast<const f32x4*>(yf + 4 * q);
        }
#pragma unroll
        for (int ii = 0; ii < 4; ++ii)
#pragma unroll
          for (int e = 0; e < 4; ++e) tr[(8 * ii + 4 * h + e) * TP + r] = acc[i][t][4 * ii + e];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const float* row = tr + (lane >> 1) * TP;
        if constexpr (EPI == 3) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(row + 16 * hf + 4 * q);
            if (live) *reinterpret_cast<f32x4*>(yf + 4 * q) = old[q] + v;
          }
        } else if constexpr (OT == 0 && EPI == 0) {
          // lane l's piece q is row 8q + l / 8, columns 4 (l % 8) .. + 4: eight
          // lanes write a whole 128-byte line of a row (the residual add above
          // is faster in the other order, its loads under one condition: 23.8 us
          // against 24.6 for 2,048 x 1,024 x 2,752)
          const int fr = m0 + i * 32 + (lane >> 3);
          float* yl = reinterpret_cast<float*>(ybase) + (int64_t)fr * p.ldy + ni[t] * 32 + 4 * (lane & 7);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(tr + (8 * q + (lane >> 3)) * TP + 4 * (lane & 7));
            f32x4* d = reinterpret_cast<f32x4*>(yl + (int64_t)(8 * q) * p.ldy);
            if (fr + 8 * q < cnt) {
              if constexpr (NTY) __builtin_nontemporal_store(v, d);
              else *d = v;
            }
          }
        } else if constexpr (EPI == 0) {
          float v0[8], v1[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) { v0[e] = row[16 * hf + e]; v1[e] = row[16 * hf + 8 + e]; }
          if (live) {
            const int64_t o = (int64_t)j * p.ldy + ni[t] * 32 + 16 * hf;
            vg_store8<OT, NTY>(ybase, o, v0);
            vg_store8<OT, NTY>(ybase, o + 8, v1);
          }
        } else {
          // hidden units ni*16 + 8*hf .. +8: gates in columns 0-15, ups in 16-31
          float v[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float g = row[8 * hf + e], u = row[16 + 8 * hf + e];
            v[e] = g / (1.0f + __expf(-g)) * u * cw;
          }
          if (live) vg_store8<OT>(ybase, (int64_t)j * p.ldy + ni[t] * 16 + 8 * hf, v);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      } else {
        // element stores: lane (r, h) holds rows 8ii + 4h + e of column r
        float up[16];
        if constexpr (EPI == 1)
#pragma unroll
          for (int e = 0; e < 16; ++e) up[e] = __shfl_xor(acc[i][t][e], 16);
        const int n = EPI == 1 ? ni[t] * 16 + r : ni[t] * 32 + r;
        const bool col = EPI == 1 ? r < 16 : n < p.N;
#pragma unroll
        for (int ii = 0; ii < 4; ++ii)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int jj = m0 + i * 32 + 8 * ii + 4 * h + e;
            if (!col || jj >= cnt) continue;
            const float a = acc[i][t][4 * ii + e];
            if constexpr (EPI == 3) {
              reinterpret_cast<float*>(ybase)[(int64_t)jj * p.ldy + n] += a;
            } else if constexpr (EPI == 0) {
              vg_store<OT>(ybase, (int64_t)jj * p.ldy + n, a);
            } else {
              float v = a / (1.0f + __expf(-a)) * up[4 * ii + e];
              if (p.comb) v *= p.comb[(p.rows ? p.rows[(int64_t)z * p.M + jj] : (int64_t)jj) * p.ldc + z];
              vg_store<OT>(ybase, (int64_t)jj * p.ldy + n, v);
            }
          }
      }
    }
  }
}

// Row lists of the routed products: expert z's rows { m : comb[m*ldc + z] != 0 }
// ascending, one workgroup per expert, 1024 rows per step (a ballot per wave,
// the waves' counts through LDS).
__global__ __launch_bounds__(1024) void k_mod_lists(const float* comb, int64_t ldc, int M, int E, int32_t* rows,
                                                    int32_t* counts, int32_t* slots) {
  __shared__ int wc[2][16];
  const int z = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int base = 0, buf = 0;
  for (int m0 = 0; m0 < M; m0 += 1024, buf ^= 1) {
    const int m = m0 + tid;
    const bool sel = m < M && comb[(int64_t)m * ldc + z] != 0.0f;
    const unsigned long long b = __ballot(sel);
    if (lane == 0) wc[buf][wave] = __popcll(b);
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int c = wc[buf][w];
      before += w < wave ? c : 0;
      total += c;
    }
    const int pos = base + before + __popcll(b & ((1ull << lane) - 1ull));
    if (sel) rows[(int64_t)z * M + pos] = m;
    if (m < M) slots[(int64_t)m * E + z] = sel ? pos : -1;
    base += total;
  }
  if (tid == 0) counts[z] = base;
}

}  // namespace

constexpr int64_t kWgLlcBytes = (int64_t)256 << 20;  // last-level cache
constexpr int kWgHeadCols = 32768;                   // an LM head's columns

int wg_run(WgParams p, int epi, int y_dtype, hipStream_t s) {
  // rows and columns are numbered to the end of their last tile in 32 bits
  if (p.M >= INT_MAX - 256 || p.N >= INT_MAX - 256) return VNX_ERR_UNSUPPORTED;
  p.nt = (int)(((int64_t)p.N + 31) / 32);
  const int ncols = epi == 1 ? p.N / 2 : p.N;
  p.vec_out = aligned16(p.y) && p.ldy % 8 == 0 && p.syb % 8 == 0 && (epi == 1 || p.N % 32 == 0) && ncols % 8 == 0;
  // Row tiles over all groups for a shape of rt 32-row tiles: all of them, and
  // as many as total_rows lets expect where counts rule.
  auto all_tiles = [&](int rt) -> int64_t { return (int64_t)p.batch * ((p.M + 32 * rt - 1) / (32 * rt)); };
  auto row_tiles = [&](int rt) -> int64_t {
    const int64_t all = all_tiles(rt), most = p.total_rows / (32 * rt) + p.batch;
    return p.counts && p.total_rows > 0 && most < all ? most : all;
  };
  auto groups = [&](int ct) { return (p.nt + 4 * ct - 1) / (4 * ct); };
  // 128 x 256 tiles where they fill two workgroups per CU, 64 x 256 where
  // those fill one, else 64 x 128 with a deeper ring.  Measured (us, in that
  // order; M rows x N x K): 16 experts, 1,024 rows each: gate-up 196 / 214 /
  // 231, 512 rows 101 / 101 / 116, down of 512 rows (256 / 512 / 1,024 tiles)
  // 71 / 66 / 68; one product: 2,048 x 5,504 x 1,024 32.3 / 28.7 / 35.9,
  // 2,048 x 2,048 x 1,024 17.2 / 13.3 / 13.9, 2,048 x 1,024 x 2,752 41 / 28 / 22.
  const int64_t cus = device_cus();
  int sh = row_tiles(4) * groups(2) >= 2 * cus ? 0 : row_tiles(2) * groups(2) >= cus ? 1 : 2;
  const int64_t wbytes = (int64_t)p.N * p.K * 2;
  if (!p.counts && p.batch == 1 && p.M > 128 && p.M <= 256 && sh != 2 && wbytes <= kWgLlcBytes) {
    // Two or fewer 128-row tiles: what counts is how many turns of the chip the
    // tiles take (2 x 128 or 3 x 64 rows a CU and turn, the latter at 1.09 times
    // the cost per row) and how much of the last row tile is empty.  129 rows x
    // 100,352 x 1,024 59 us by the rule above, 48; 224 x 64,000 x 1,024 39 and 35.  A
    // W that the last-level cache cannot hold is read once per row tile: 129 x
    // 248,320 x 1,024 145 with two, 148 with three.
    const int64_t turns0 = (row_tiles(4) * groups(2) + 2 * cus - 1) / (2 * cus);
    const int64_t turns1 = (row_tiles(2) * groups(2) + 3 * cus - 1) / (3 * cus);
    sh = row_tiles(4) * groups(2) > cus && turns0 * 256 <= turns1 * 209 ? 0 : 1;
  }
  // The launch covers all rows whatever total_rows says: how many rows the
  // lists hold is the device's to know (a row whose router logits are NaN is on
  // every expert's), and the workgroups past the live tiles return at once (a
  // prefill of 4 x 512 tokens with one MoD layer: 875 us, as when the launch
  // was cut to the expected rows).
  const int64_t tiles = sh == 0 ? all_tiles(4) * groups(2) : sh == 1 ? all_tiles(2) * groups(2)
                                                                      : all_tiles(2) * groups(1);
  p.ng = groups(sh == 2 ? 1 : 2);
  const int64_t wgs = (tiles + kVgXcds - 1) / kVgXcds * kVgXcds;
  if (wgs >= INT_MAX) return VNX_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)wgs);
  // One row tile reads each byte of W once.  A W that the last-level cache cannot
  // hold then leaves nothing there that this launch or the next would read
  // again, and pushes out what the other layers read, so it streams past the
  // caches: 128 rows x 200,064 x 1,024 101 -> 93 us, 8 x 151,936 x 2,048 120 -> 110,
  // and a 4-layer verify of 8 x 7 tokens around the 248,320 x 1,024 head 344 ->
  // 330.  One that fits is better left there (64 rows x 131,072 x 512 28.7 us
  // streamed, 25.0 not; x 1,024, the whole cache, 49.6 and 45.1).
  // From two row tiles on the second read has to hit: at 224 rows of the
  // 248,320 head 143 us cached, 181 streamed.
  const bool nt = p.M <= 128 && wbytes > kWgLlcBytes;
  // Logits past the caches (a head's columns): fp32 ones always, as they come in
  // whole lines (128 rows x 32,768 x 1,024 14.3 us, 15.6 through the caches); 16-bit
  // ones where they would push out a W that the caches hold between two calls
  // (224 rows x 64,000 x 2,048 68 us, 85), and not otherwise: the kernel that
  // reads them next finds them there.
  const int64_t obytes = (int64_t)p.M * p.N * (y_dtype == VNX_F32 ? 4 : 2);
  const bool nty = p.N >= kWgHeadCols &&
                   (y_dtype == VNX_F32 || (wbytes <= kWgLlcBytes && wbytes + obytes > kWgLlcBytes / 4 * 3));
  auto shape = [&](auto ot, auto ep) -> int {
    constexpr int OT = decltype(ot)::value, EP = decltype(ep)::value;
    auto go = [&](auto cp) {
      constexpr int CP = decltype(cp)::value;
      if (sh == 0) hipLaunchKernelGGL((k_wgemm<OT, EP, 4, 2, 1, 2, 2, CP>), grid, dim3(256), 0, s, p);
      else if (sh == 1) hipLaunchKernelGGL((k_wgemm<OT, EP, 2, 2, 1, 1, 3, CP & kWgNtY>), grid, dim3(256), 0, s, p);
      else hipLaunchKernelGGL((k_wgemm<OT, EP, 2, 1, 2, 4, 2, CP & kWgNtY>), grid, dim3(256), 0, s, p);
    };
    constexpr int W = EP == 0 ? kWgNtW : 0, Y = EP == 0 ? kWgNtY : 0;
    if (EP == 0 && sh == 0 && nt && nty) go(IntC<W | Y>{});
    else if (EP == 0 && sh == 0 && nt) go(IntC<W>{});
    else if (EP == 0 && nty) go(IntC<Y>{});
    else go(IntC<0>{});
    VNX_LAUNCH_CHECK();
    return VNX_OK;
  };
  if (epi == 3) return shape(IntC<0>{}, IntC<3>{});
  auto by_epi = [&](auto ot) -> int { return epi == 1 ? shape(ot, IntC<1>{}) : shape(ot, IntC<0>{}); };
  if (y_dtype == VNX_F32) return by_epi(IntC<0>{});
  if (y_dtype == VNX_BF16) return by_epi(IntC<1>{});
  return by_epi(IntC<2>{});
}

}  // namespace vnx

using namespace vnx;

extern "C" {

int vnx_mod_lists(const float* comb, int64_t ldc, int64_t M, int experts, int32_t* rows, int32_t* counts,
                  int32_t* slots, void* stream) {
  if (!comb || !rows || !counts || !slots || M < 0 || experts < 1 || ldc < experts) return VNX_ERR_INVALID_ARG;
  if (M >= INT_MAX - 1024 || experts > 65535) return VNX_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(k_mod_lists, dim3((unsigned)experts), dim3(1024), 0, static_cast<hipStream_t>(stream), comb, ldc,
                     (int)M, experts, rows, counts, slots);
  VNX_LAUNCH_CHECK();
  return VNX_OK;
}

int vnx_expert_gemm_bf16_rows(const void* x, int64_t ldx, int64_t sxb, const void* w_packed, int64_t swb, int64_t M,
                              int64_t N, int64_t K, int experts, int epilogue, const float* comb, int64_t ldc,
                              const int32_t* rows, const int32_t* counts, int64_t total_rows, void* y, int y_dtype,
                              int64_t ldy, int64_t syb, void* stream) {
  if (!x || !w_packed || !y || !counts || M < 0 || N < 0 || K <= 0 || experts < 0 || total_rows < 0)
    return VNX_ERR_INVALID_ARG;
  if (epilogue != VNX_EPI_NONE && epilogue != VNX_EPI_SWIGLU) return VNX_ERR_INVALID_ARG;
  if (y_dtype != VNX_F32 && y_dtype != VNX_BF16 && y_dtype != VNX_F16) return VNX_ERR_UNSUPPORTED;
  const bool sw = epilogue == VNX_EPI_SWIGLU;
  if (ldx < K || ldy < (sw ? N / 2 : N) || sxb < 0 || swb < 0 || syb < 0) return VNX_ERR_INVALID_ARG;
  if (experts > 1 && swb < (N + 31) / 32 * 32 * K) return VNX_ERR_INVALID_ARG;
  if (sw && N % 32) return VNX_ERR_INVALID_ARG;
  if (comb && (!sw || ldc < experts)) return VNX_ERR_INVALID_ARG;
  if (M == 0 || N == 0 || experts == 0) return VNX_OK;
  if (K % kVgChunk || ldx % 8 || sxb % 8 || swb % 8 || !aligned16(x) || !aligned16(w_packed))
    return VNX_ERR_UNSUPPORTED;
  if (M >= INT_MAX || N >= INT_MAX || K >= INT_MAX) return VNX_ERR_UNSUPPORTED;
  WgParams p{};
  p.x = static_cast<const uint16_t*>(x); p.w = static_cast<const uint16_t*>(w_packed); p.y = y; p.comb = comb;
  p.rows = rows; p.counts = counts; p.total_rows = total_rows;
  p.ldx = ldx; p.sxb = sxb; p.swb = swb; p.ldy = ldy; p.syb = syb; p.ldc = ldc;
  p.M = (int)M; p.N = (int)N; p.K = (int)K; p.batch = experts;
  return wg_run(p, epilogue, y_dtype, static_cast<hipStream_t>(stream));
}

}  // extern "C"
