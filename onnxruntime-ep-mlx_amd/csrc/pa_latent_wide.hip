// pa_latent_wide.hip -- the LATENT layout's MLA rows (576 key dims, values = the first 512) against
// blocks of 64 grouped query rows, on gfx950 matrix cores.
//
// (The reference's latent route: attention.rs:4058-4062, :4210-4213.)  One workgroup of four
// wavefronts, one per SIMD, takes steps of 64 keys:
//   S^T = K . Q^T    wavefront w: rows 32 (w % 2) .., keys 32 (w / 2) ..; A = 32 keys x 16 dims from
//                    LDS, B = its rows' queries (144 registers), a lane holds one row's 16 scores.
//   softmax          row maxima of the two key halves are exchanged through LDS; the probabilities,
//                    split into hi + lo parts as everywhere, go to LDS as the next product's operand.
//   O^T += V^T . P^T wavefront w: value dims 128 w .. of all 64 rows; A = 32 dims x 16 keys: a lane
//                    reads 8 bytes (4 dims) of 8 rows and regroups them with byte permutes, so row m
//                    of tile j is value dim 128 w + 4 m + j.
// Every operand read from LDS feeds 32x32x16 products, and a row leaves L2 once per 64 query rows.
// Steps go through two LDS slots (147 KB) by direct loads of whole lines, one in flight while the
// other is computed; 16-byte piece x of row r sits at x ^ ((r / 2) % 8) of its group of 8, so the 16
// rows of a key operand read meet 16 different bank groups (a row is 1152 bytes: its parity picks
// the half).  The lo parts take the place of the step's dims 512 .. 575, which only scores read.
// Work: the steps of all (row block, sequence) pairs in order, in equal segments, one per workgroup
// (and CU).  Row blocks come outermost: the blocks of one sequence run at the same time, half a grid
// apart (on the same XCD), and share its rows in L2.  A pair inside one segment writes its rows; one
// that meets several leaves a partial in each (slot 2 segment + 1 where it starts, 2 segment after
// that) for latent_merge_kernel.
// Bound by matrix-core and LDS issue: 100 products of 32 cycles per wavefront and step against 69 KB
// it reads from LDS.   128 heads over 64 contexts of 512 .. 8192
// keys (320 K keys, 369 MB): 190 us, 1.9 TB/s of rows and 30 % of the cycles on matrix products, against
// 524 us in 32-row blocks by latent_kernel; measured on the way: all loads of a step issued at its start
// 203 us, key operands read one product ahead only 213.
//
// Compiled with -amdgpu-mfma-vgpr-form (Makefile): accumulators in ordinary registers, the queries in
// the accumulation half of the file.  With accumulators there the compiler moves all 128 of a lane
// both ways in every step, for the rescale that few steps take.
#include <algorithm>
#include <type_traits>

#include "pa_tiles.hpp"

namespace pa {
namespace {

constexpr int kWideD = 576, kWideVD = kLatWideDims, kWideRows = kLatWideRows, kWideKeys = 64;
constexpr int kWideKs = kWideD / 16, kWideCpr = kWideD / 8;  // 16-dim k-steps, 16-byte pieces per row
constexpr int kWideRowB = kWideD * 2, kWideSlotB = kWideKeys * kWideRowB;
constexpr int kWideMaxPairs = 4096;  // every workgroup scans the pairs

typedef float f32x16 __attribute__((ext_vector_type(16)));
template <typename TT>
__device__ __forceinline__ f32x16 wide_mfma(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (TT::code == PA_DTYPE_FLOAT16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float other_half(float x) {  // lane l ^ 32's x
  return __shfl_xor(x, 32, 64);
}

// One direct LDS load: 16 bytes per lane from base + off to LDS byte address lds + 16 * lane.  As
// inline assembly, so that the compiler's memory counters do not see it and nothing waits for it but
// the step loop.  (M0, the LDS base, is reserved: the compiler sets it before each use of its own.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(off), "s"(base), "s"(lds)
               : "memory", "m0");
}
#pragma clang diagnostic pop

// A (row block, sequence) pair: its rows, first key and end of the rows it reads, 64-key steps.
struct WidePair {
  int rb, b, s0, nq, pastb, total, t_first, t_end, n;
};
__device__ __forceinline__ WidePair wide_pair(const AttnParams& p, int e, int rbs) {
  WidePair q{};
  const bool live = e < p.batch * rbs;
  q.rb = live ? e / p.batch : 0;
  q.b = live ? e - q.rb * p.batch : 0;
  const int c0 = p.cum[q.b], c1 = p.cum[q.b + 1];
  q.s0 = min(max(c0, 0), p.num_tokens);
  q.nq = min(max(c1, q.s0), p.num_tokens) - q.s0;
  const int H = p.num_heads, row0 = q.rb * kWideRows;
  if (!live || (int64_t)row0 >= (int64_t)H * q.nq) return q;
  q.pastb = clamped_past(p, q.b, q.nq);
  q.total = seq_total(p, q.b, q.pastb, q.nq);
  const int r_last = (int)min((int64_t)row0 + kWideRows, (int64_t)H * q.nq) - 1;
  const int hi = min(q.total, p.causal ? q.pastb + r_last / H + 1 : q.total);
  const int lo = p.window > 0 ? max(0, q.pastb + row0 / H - p.window + 1) : 0;
  q.t_first = lo < hi ? (lo / 32) * 32 : 0;  // (no row sees a key: one masked step)
  q.t_end = min(q.total, q.t_first + (max(hi - q.t_first, 1) + 31) / 32 * 32);
  q.n = (q.t_end - q.t_first + kWideKeys - 1) / kWideKeys;
  return q;
}
__device__ __forceinline__ int wide_scan(int v, int lane) {  // inclusive, over the wavefront
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  return v;
}
// Steps of all pairs; head: the lane's pair of the first 64.
__device__ __forceinline__ int wide_steps(const AttnParams& p, int rbs, int lane,
                                          const WidePair& head) {
  int n = head.n;
#pragma unroll 2
  for (int base = 64; base < p.batch * rbs; base += 64) n += wide_pair(p, base + lane, rbs).n;
  return __builtin_amdgcn_readlane(wide_scan(n, lane), 63);
}
// Segment i of g covers the steps [i S / g, (i + 1) S / g): as few segments as keep the longest at
// ceil(S / grid) steps (320 steps in 256 segments cut most pairs once more for nothing).
__device__ __forceinline__ int wide_segments(int S, int grid) {
  const int L = max(1, (S + grid - 1) / grid);
  return max(1, (S + L - 1) / L);
}
__device__ __forceinline__ int wide_seg_of(int step, int S, int g) {
  return (int)((((int64_t)step + 1) * g - 1) / S);
}

template <typename TT, bool CAP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void
latent_wide_kernel(const AttnParams p, int rbs) {
  using vec8 = typename TT::vec8;
  __shared__ u32x4 ring[2 * kWideSlotB / 16];
  __shared__ u32x4 phi[4][2][64];  // [16-key chunk][row tile][lane]
  __shared__ float mx[2][64];      // [key half][row]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int rt = wave & 1, kh = wave >> 1;
  const int H = p.num_heads, E = p.batch * rbs;
  const WidePair head = wide_pair(p, lane, rbs);
  const int S = wide_steps(p, rbs, lane, head);
  const int nseg = wide_segments(S, gridDim.x), seg = blockIdx.x;
  // The merge's list: a pair's rows and segments, its first row, its sequence's first token, its first
  // segment.  With fewer pairs than segments an entry per pair, all written by segment 0; else an
  // entry per segment for the pair that it starts and does not finish.
  int4* const info = reinterpret_cast<int4*>(p.plan_info);
  const bool per_pair = E < (int)gridDim.x;
  auto entry = [&](int rows, int row0, int s0, int P, int n) {
    const int f = wide_seg_of(P, S, nseg);
    return make_int4(rows | ((wide_seg_of(P + n - 1, S, nseg) - f + 1) << 8), row0, s0, f);
  };
  if (per_pair && seg == 0 && threadIdx.x < 64) {
    for (int base = 0, carry = 0; base < E; base += 64) {
      const WidePair q = base ? wide_pair(p, base + lane, rbs) : head;
      const int incl = wide_scan(q.n, lane), row0 = q.rb * kWideRows;
      if (base + lane < E)
        info[base + lane] = q.n > 0 ? entry(min(H * q.nq - row0, kWideRows), row0, q.s0,
                                            carry + incl - q.n, q.n)
                                    : make_int4(0, 0, 0, 0);
      carry += __builtin_amdgcn_readlane(incl, 63);
    }
  }
  if (!per_pair && threadIdx.x == 0) info[seg] = make_int4(0, 0, 0, 0);
  if (S <= 0 || seg >= nseg) return;
  const int gs = (int)((int64_t)seg * S / nseg), ge = (int)(((int64_t)seg + 1) * S / nseg);

  const uint32_t qxor = p.scale < 0.0f ? 0x80008000u : 0u;
  const float scale = fabsf(p.scale), scale_log2 = fabsf(p.scale_log2);
  const float cap_k = CAP ? scale / p.softcap : 0.0f, cap_l2 = p.softcap * kLog2e;
  char* const lbase = reinterpret_cast<char*>(&ring[0]);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lbase;
  // Direct loads: wavefront w fetches the 16 rows 16 w .. of a step, 18 loads of 64 pieces.
  // Load 9 + i fetches the pieces of load i from 8 rows on.
  constexpr int NIH = 8 * kWideCpr / 64;
  uint32_t poff[NIH];  // byte offset of the lane's piece from the first of the 16 rows
#pragma unroll
  for (int i = 0; i < NIH; ++i) {
    const int s = 64 * i + lane, r = s / kWideCpr, x = s % kWideCpr;
    poff[i] = r * kWideRowB + 16 * (x ^ (r >> 1));
  }
  // Operand addresses in a slot.  Keys: row 32 kh + c, piece 2 ks + h; values: rows 4 h + (q % 4) +
  // 8 (q / 4) of a 16-key chunk, piece 16 wave + c / 2.
  int kofs[4], vofs[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    kofs[i] = (32 * kh + c) * kWideRowB + 16 * ((2 * i + h) ^ ((c >> 1) & 7));
    const int r = 4 * h + 2 * (i & 1) + 8 * (i >> 1);
    vofs[i] = r * kWideRowB + 16 * ((16 * wave + (c >> 1)) ^ ((r >> 1) & 7)) + 8 * (c & 1);
  }
  // lo part of P: 16-byte piece l of chunk t and row tile j in the tail of row 8 (2 t + j) + l / 8
  const int tofs = (lane >> 3) * kWideRowB + 2 * kWideVD + 16 * (lane & 7);

  int carry = 0;
  for (int base = 0; base < E && carry < ge; base += 64) {
    const WidePair mine = base ? wide_pair(p, base + lane, rbs) : head;
    const int incl = wide_scan(mine.n, lane);
    const int first = carry + incl - mine.n;  // first step of the lane's pair in the list
    uint64_t todo = __ballot(mine.n > 0 && first < ge && first + mine.n > gs);
    carry += __builtin_amdgcn_readlane(incl, 63);
    while (todo) {
      const int l = __builtin_ctzll(todo);
      todo &= todo - 1;
      auto of = [&](int v) { return __builtin_amdgcn_readlane(v, l); };
      const int P = of(first), n = of(mine.n), b = of(mine.b), s0 = of(mine.s0);
      const int nq = of(mine.nq), pastb = of(mine.pastb), total = of(mine.total);
      const int row0 = of(mine.rb) * kWideRows, R = H * nq, t_end = of(mine.t_end);
      const int k0 = max(gs - P, 0), k1 = min(ge - P, n);
      const int t_first = of(mine.t_first) + kWideKeys * k0, nsteps = k1 - k0;
      const bool whole = k0 == 0 && k1 == n;
      if (!per_pair && k0 == 0 && k1 < n && threadIdx.x == 0)
        info[seg] = entry(min(R - row0, kWideRows), row0, s0, P, n);

      const WaveInfo w = make_wave(p, kWideD, b, 0, s0, pastb, total);
      PageWindow pw;
      window_at(pw, w, min(div_bs(t_first, w), w.max_blocks - 1), lane);
      const char* last_row;  // read again by rows past the pair's end
      {
        int64_t blk = w.bt[min(div_bs(t_end - 1, w), w.max_blocks - 1)];
        blk = min(max(blk, (int64_t)0), w.num_blocks - 1);
        last_row = w.kc + (blk * w.bs + mod_bs(t_end - 1, w)) * w.rowb;
      }
      // this lane's query row for the scores
      const int r = row0 + 32 * rt + c;
      const bool rvalid = r < R;
      const int qi = rvalid ? r / H : 0, head = rvalid ? r % H : 0;
      const int rpos = pastb + qi;
      const int vis_lo = p.window > 0 ? rpos - p.window + 1 : 0;
      const int vis_hi = rvalid ? min(total, p.causal ? rpos + 1 : total) : -1;
      // keys every row of the tile sees (none with rows past R)
      int all_lo = 0, all_hi = -1;
      if (row0 + 32 * rt + 32 <= R) {
        const int qf = (row0 + 32 * rt) / H, ql = (row0 + 32 * rt + 31) / H;
        all_hi = min(total, p.causal ? pastb + qf + 1 : total);
        all_lo = p.window > 0 ? pastb + ql - p.window + 1 : 0;
      }
      u32x4 qv[kWideKs];  // (zero for rows past R: scores of 0, masked)
      {
        const char* qrow = reinterpret_cast<const char*>(p.q) +
                           (((int64_t)(s0 + qi) * H + head) * kWideD + 8 * h) * 2;
        const uint32_t qmask = rvalid ? ~0u : 0u;
#pragma unroll
        for (int ks = 0; ks < kWideKs; ++ks)
          qv[ks] = (ld16(qrow + 32 * ks) ^ qxor) & qmask;
      }
      f32x16 o[2][4];
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[j >> 2][j & 3][i] = 0.0f;
      float m_run[2] = {kNegInf, kNegInf}, l_part = 0.0f;  // of rows c and 32 + c; of row r

      // Rows of step k to its slot: where this wavefront's 16 come from and go, whole or with rows past
      // the end, which read the last row of the tile before it, or the pair's last row.
      const char* tb;
      uint32_t dst;
      auto locate = [&](int k) __attribute__((always_inline)) {
        const int t = t_first + kWideKeys * k + 16 * wave;
        const int bi = min(div_bs(t, w), w.max_blocks - 1);
        if (bi < pw.first || bi >= pw.first + 64) window_at(pw, w, bi, lane);
        int64_t blk = __builtin_amdgcn_readlane(pw.ids, bi - pw.first);
        blk = min(max(blk, (int64_t)0), w.num_blocks - 1);
        tb = w.kc + (blk * w.bs + mod_bs(t, w)) * w.rowb;
        dst = __builtin_amdgcn_readfirstlane(lds0 + (k & 1) * kWideSlotB + wave * (16 * kWideRowB));
        return t + 16 <= t_end;
      };
      auto load = [&](int i) __attribute__((always_inline)) {
        dma16(i < NIH ? tb : tb + 8 * kWideRowB, i < NIH ? poff[i] : poff[i - NIH] ^ 64u,
              dst + 1024 * i);
      };
      auto load_tail = [&](int k) __attribute__((always_inline)) {
        const int t = t_first + kWideKeys * k + 16 * wave;
        const char* base = t < t_end ? tb : last_row;
        const int keep = t < t_end ? t_end - t - 1 : 0;
        for (int i = 0; i < 2 * NIH; ++i) {
          const int s = 64 * i + lane, rr = s / kWideCpr, x = s % kWideCpr;
          dma16(base, min(rr, keep) * kWideRowB + 16 * (x ^ ((rr >> 1) & 7)), dst + 1024 * i);
        }
      };
      // Scores of the slot at sb, the next step's loads among the products (LOADS): all at once they
      // hold up the wavefront for as long as the address unit takes for them.
      auto product = [&](auto LOADS, const char* sb, f32x16& sc) __attribute__((always_inline)) {
        f32x16 sd;
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = sd[i] = 0.0f;
        // operands read kAhead k-steps ahead; the fences keep the compiler from pulling the reads
        // back to their products, each of which then waits out the LDS latency
        constexpr int kAhead = 6;
        u32x4 kx[kAhead];
        auto key = [&](int ks) __attribute__((always_inline)) {
          return *reinterpret_cast<const u32x4*>(sb + kofs[ks & 3] + 128 * (ks >> 2));
        };
#pragma unroll
        for (int ks = 0; ks < kAhead; ++ks) kx[ks] = key(ks);
#pragma unroll
        for (int ks = 0; ks < kWideKs; ++ks) {
          __builtin_amdgcn_sched_barrier(0);
          if (ks & 1)
            sd = wide_mfma<TT>(kx[ks % kAhead], qv[ks], sd);
          else
            sc = wide_mfma<TT>(kx[ks % kAhead], qv[ks], sc);
          if (ks + kAhead < kWideKs) kx[ks % kAhead] = key(ks + kAhead);
          if constexpr (decltype(LOADS)::value)
            if (ks & 1) load(ks >> 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        sc += sd;
      };

      __syncthreads();  // the previous pair's LDS has been read
      if (locate(0)) {
#pragma unroll
        for (int i = 0; i < 2 * NIH; ++i) load(i);
      } else {
        load_tail(0);
      }
      for (int k = 0; k < nsteps; ++k) {
        __builtin_amdgcn_s_waitcnt(0x0F70);  // this wavefront's loads of step k
        __syncthreads();                     // everyone's; and step k - 1 has been read
        char* const sb = lbase + (k & 1) * kWideSlotB;
        float x[16];
        {
          f32x16 sc;
          const bool more = k + 1 < nsteps;
          if (more && locate(k + 1)) {
            product(std::true_type{}, sb, sc);
          } else {
            if (more) load_tail(k + 1);
            product(std::false_type{}, sb, sc);
          }
#pragma unroll
          for (int i = 0; i < 16; ++i)
            x[i] = CAP ? softcap_log2(sc[i], cap_k, cap_l2) : sc[i] * scale_log2;
          const int t0 = t_first + kWideKeys * k + 32 * kh;
          if (!(t0 >= all_lo && t0 + 32 <= all_hi)) {
            // positions [vis_lo, vis_hi) of the row, one unsigned range test per score
            const unsigned span = vis_hi > vis_lo ? (unsigned)vis_hi - (unsigned)vis_lo : 0u;
            const unsigned rel = (unsigned)(t0 + 4 * h) - (unsigned)vis_lo;
#pragma unroll
            for (int i = 0; i < 16; ++i)
              x[i] = (rel + 8 * (i >> 2) + (i & 3) < span) ? x[i] : kNegInf;
          }
          float lmax = x[0];
#pragma unroll
          for (int i = 1; i < 16; ++i) lmax = fmaxf(lmax, x[i]);
          lmax = fmaxf(lmax, other_half(lmax));
          if (h == 0) mx[kh][32 * rt + c] = lmax;
        }
        __syncthreads();
        {
          // the lazy rescale of the other kernels, decided alike by every wavefront
          const float a0 = fmaxf(mx[0][c], mx[1][c]);
          const float a1 = fmaxf(mx[0][32 + c], mx[1][32 + c]);
          if (__any(a0 > m_run[0] + 8.0f || a1 > m_run[1] + 8.0f)) {
            float alpha[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const float m_new = fmaxf(m_run[j], j ? a1 : a0);
              alpha[j] = (m_run[j] == kNegInf || m_new == kNegInf) ? 1.0f : exp2f(m_run[j] - m_new);
              m_run[j] = m_new;
#pragma unroll
              for (int q = 0; q < 4; ++q) o[j][q] *= alpha[j];
            }
            l_part *= rt ? alpha[1] : alpha[0];
          }
        }
        {
          const float m = rt ? m_run[1] : m_run[0], msafe = m == kNegInf ? 0.0f : m;
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            float pv[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              pv[i] = __builtin_amdgcn_exp2f(x[8 * t + i] - msafe);
              l_part += pv[i];
            }
            vec8 hi8, lo8;
            TT::split8(pv, hi8, lo8);
            phi[2 * kh + t][rt][lane] = __builtin_bit_cast(u32x4, hi8);
            *reinterpret_cast<u32x4*>(sb + tofs + 8 * (2 * (2 * kh + t) + rt) * kWideRowB) =
                __builtin_bit_cast(u32x4, lo8);
          }
        }
        __syncthreads();
        // operands of a 16-key chunk, read one chunk ahead
        struct Chunk {
          u32x4 ph[2], pl[2];
          u32x2 v[8];
        } ch[2];
        auto read = [&](Chunk& d, int t) __attribute__((always_inline)) {
#pragma unroll
          for (int q = 0; q < 8; ++q)
            d.v[q] = *reinterpret_cast<const u32x2*>(sb + vofs[q >> 1] +
                                                     (16 * t + (q & 1)) * kWideRowB);
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            d.ph[j] = phi[t][j][lane];
            d.pl[j] = *reinterpret_cast<const u32x4*>(sb + tofs + 8 * (2 * t + j) * kWideRowB);
          }
        };
        read(ch[0], 0);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          __builtin_amdgcn_sched_barrier(0);
          if (t < 3) read(ch[(t + 1) & 1], t + 1);
          const Chunk& d = ch[t & 1];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            u32x4 a;
#pragma unroll
            for (int m = 0; m < 4; ++m)
              a[m] = __builtin_amdgcn_perm(d.v[2 * m + 1][j >> 1], d.v[2 * m][j >> 1],
                                           (j & 1) ? 0x07060302u : 0x05040100u);
            o[0][j] = wide_mfma<TT>(a, d.ph[0], o[0][j]);
            o[1][j] = wide_mfma<TT>(a, d.ph[1], o[1][j]);
            o[0][j] = wide_mfma<TT>(a, d.pl[0], o[0][j]);
            o[1][j] = wide_mfma<TT>(a, d.pl[1], o[1][j]);
          }
        }
      }

      // sums of both key halves
      const float l_row = l_part + other_half(l_part);
      __syncthreads();
      if (h == 0) mx[kh][32 * rt + c] = l_row;
      __syncthreads();
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int ro = row0 + 32 * j + c;
        if (ro >= R) continue;
        const float l_sum = mx[0][32 * j + c] + mx[1][32 * j + c];
        if (whole) {
          const int hd = ro % H;
          const float f = finalize_factor(m_run[j], l_sum, sink_logit<TT>(p, hd));
          typename TT::raw* dst = reinterpret_cast<typename TT::raw*>(p.out) +
                                  ((int64_t)(s0 + ro / H) * H + hd) * kWideVD + 128 * wave;
#pragma unroll
          for (int i = 0; i < 16; i += 2) {
            u32x4 pk;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
              const int u = i + (m >> 1), q = 2 * (m & 1);
              pk[m] = (uint32_t)TT::from_f32(o[j][q][u] * f) |
                      ((uint32_t)TT::from_f32(o[j][q + 1][u] * f) << 16);
            }
            *reinterpret_cast<u32x4*>(dst + 4 * (8 * (i >> 2) + 4 * h + (i & 3))) = pk;
          }
        } else {
          const int64_t row = (int64_t)(2 * seg + (k0 == 0)) * kWideRows + 32 * j + c;
          float* dst = p.part_o + row * kWideVD + 128 * wave;
#pragma unroll
          for (int i = 0; i < 16; ++i)
            *reinterpret_cast<f32x4*>(dst + 4 * (8 * (i >> 2) + 4 * h + (i & 3))) =
                f32x4{o[j][0][i], o[j][1][i], o[j][2][i], o[j][3][i]};
          if (h == 0 && wave == 0) {
            p.part_ml[row * 2 + 0] = m_run[j];
            p.part_ml[row * 2 + 1] = l_sum;
          }
        }
      }
    }
  }
}

// Merge the partials of entry blockIdx.y of the list where the pair spans segments: one workgroup per
// row, four output dims per thread, GR groups of 128 threads with every GR-th partial each, four in
// flight.  Bound by the latency of those rounds where few pairs share the segments (one row block
// spans up to 128): four groups there.   128 heads, 64 sequences (384
// partials, 50 MB): 11.8 us; finding the pairs again in each workgroup instead of the list 33.
template <typename TT, int GR>
__global__ __launch_bounds__(128 * GR) void latent_merge_kernel(const AttnParams p) {
  const int rl = blockIdx.x, H = p.num_heads;
  const int tid = threadIdx.x & 127, gr = threadIdx.x >> 7;
  const int4 info = reinterpret_cast<const int4*>(p.plan_info)[blockIdx.y];
  const int r = info.y + rl, s0 = info.z, seg = info.w, nparts = info.x >> 8;
  if (rl >= (info.x & 255) || nparts < 2) return;
  constexpr int U = 4;
  float M = kNegInf, lsum = 0.0f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  auto add = [&](float m, float l, f32x4 v, float mn) {
    const float wt = m != kNegInf ? exp2f(m - mn) : 0.0f;
    lsum += l * wt;
    acc += v * wt;  // also at weight 0: the row is NaN where the partial's scores are
  };
  for (int k0 = gr; k0 < nparts; k0 += U * GR) {
    float2 ml[U];
    f32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + u * GR, nparts - 1);
      const int64_t row = (int64_t)(2 * (seg + k) + (k == 0)) * kWideRows + rl;
      ml[u] = reinterpret_cast<const float2*>(p.part_ml)[row];
      v[u] = *reinterpret_cast<const f32x4*>(p.part_o + row * kWideVD + 4 * tid);
    }
    float mn = M;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k0 + u * GR < nparts) mn = fmaxf(mn, ml[u].x);
    const float a = (M == kNegInf) ? 0.0f : exp2f(M - mn);
    lsum *= a;
    acc *= a;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k0 + u * GR < nparts) add(ml[u].x, ml[u].y, v[u], mn);
    M = mn;
  }
  if constexpr (GR > 1) {
    __shared__ f32x4 sh_o[GR - 1][128];
    __shared__ float2 sh_ml[GR];
    if (gr > 0) sh_o[gr - 1][tid] = acc;
    if (tid == 0) sh_ml[gr] = make_float2(M, lsum);
    __syncthreads();
    if (gr > 0) return;
    float mn = M;
#pragma unroll
    for (int g = 1; g < GR; ++g) mn = fmaxf(mn, sh_ml[g].x);
    const float a = (M == kNegInf) ? 0.0f : exp2f(M - mn);
    lsum *= a;
    acc *= a;
#pragma unroll
    for (int g = 1; g < GR; ++g) add(sh_ml[g].x, sh_ml[g].y, sh_o[g - 1][tid], mn);
    M = mn;
  }
  const int head = r % H;
  const float fct = finalize_factor(M, lsum, sink_logit<TT>(p, head));
  u32x2 pk;
#pragma unroll
  for (int m = 0; m < 2; ++m)
    pk[m] = (uint32_t)TT::from_f32(acc[2 * m] * fct) |
            ((uint32_t)TT::from_f32(acc[2 * m + 1] * fct) << 16);
  *reinterpret_cast<u32x2*>(reinterpret_cast<typename TT::raw*>(p.out) +
                            ((int64_t)(s0 + r / H) * H + head) * kWideVD + 4 * tid) = pk;
}

template <typename TT>
void launch_wide_t(const AttnParams& p, int rbs, int grid, hipStream_t s) {
  if (p.softcap > 0.0f)
    hipLaunchKernelGGL((latent_wide_kernel<TT, true>), dim3(grid), dim3(256), 0, s, p, rbs);
  else
    hipLaunchKernelGGL((latent_wide_kernel<TT, false>), dim3(grid), dim3(256), 0, s, p, rbs);
  const int pairs = p.batch * rbs;
  const dim3 mgrid(kWideRows, std::min(pairs, grid));
  if (pairs * 8 <= grid)
    hipLaunchKernelGGL((latent_merge_kernel<TT, 4>), mgrid, dim3(512), 0, s, p);
  else
    hipLaunchKernelGGL((latent_merge_kernel<TT, 1>), mgrid, dim3(128), 0, s, p);
}

}  // namespace

// MLA shapes of the wide kernel: its row size, whole 16-key tiles per page; 32-bit step counts.
bool latent_wide_supported(int head_dim, int v_head_dim, pa_dtype act, pa_dtype cache_dtype,
                           int block_size, int max_blocks, int batch, int64_t rbs) {
  return latent_mfma_supported(head_dim, v_head_dim, act, cache_dtype) && head_dim == kWideD &&
         v_head_dim == kWideVD && block_size % 16 == 0 && max_blocks > 0 && batch > 0 && rbs >= 1 &&
         batch * rbs <= kWideMaxPairs &&
         ((int64_t)max_blocks * block_size / kWideKeys + 2) * batch * rbs < (int64_t)INT32_MAX;
}

hipError_t launch_latent_wide(const AttnParams& p, pa_dtype act, pa_dtype cache_dtype,
                              hipStream_t s) {
  if (p.batch <= 0 || p.num_tokens <= 0) return hipSuccess;
  const int mq = p.max_query_len > 0 ? p.max_query_len : p.num_tokens;
  const int64_t rbs = latent_wide_row_blocks(p.num_heads, mq);
  if (!latent_wide_supported(p.head_dim, p.v_head_dim, act, cache_dtype, p.block_size, p.max_blocks,
                             p.batch, rbs) ||
      p.kv_heads != 1 || !p.v_from_key || !p.new_rows_in_cache || !p.part_o || !p.plan_info || p.max_splits < 1 ||
      p.block_size < 16)
    return hipErrorInvalidValue;
  if (act == PA_DTYPE_FLOAT16)
    launch_wide_t<TF16>(p, (int)rbs, p.max_splits, s);
  else
    launch_wide_t<TBF16>(p, (int)rbs, p.max_splits, s);
  return hipGetLastError();
}

}  // namespace pa
