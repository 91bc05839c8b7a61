// The split-operand convolution onto up to 32 output planes, and up to 48 on small levels: a wavefront owns its rows from the rule to the store.  The
// arithmetic is that of conv_split.hip, to the bit where the additions come in the same order; see conv.hip for the family.
#include "conv_common.h"

namespace scn {

// A wavefront owns GW granules (16 positions each) and NCB column blocks, and shares nothing with the others of its workgroup,
// so that nothing waits at a barrier in the loop.  Per (slab of 32 input channels, tap) iteration:
//   indices          two iterations ahead, straight from the table (16 consecutive entries per granule)
//   gathered rows    an iteration ahead, four lanes reading 64 consecutive bytes of a row, turned into operand order through
//                    2 KB of LDS per granule that only this wavefront touches, then split in registers: once per row and
//                    tap, since no other wavefront needs it
//   weights          requested behind the MFMAs of the iteration before, from L2 in operand order, once for all GW granules
//   MFMAs            six per granule and column block, granules without the tap skipped by the table's masks
// PAIR (up to 16 input channels): an iteration is two taps of 16 channels instead of one of 32; half an operand comes from
// either, rows and weights alike.
// DEAL = 4 or 8: the wavefronts of a workgroup share GW granules and take the iterations in turn; their sums meet in LDS and are
// added in the wavefronts' order.  A small level is as long as one wavefront's chain of iterations, and this cuts it to a
// quarter without partial sums in memory and a launch to add them up.  (A cursor finds its tap by one lane read: walking the bits of
// a mask tap by tap, eight wavefronts spent more on that than on the rest: 1.6 k sites 48 -> 48 9.7 us, 7.8 so.)
// What bounds it: at large levels the vector instructions of the splitting (some 60 per granule and iteration) next to the
// MFMAs: in a loop of nothing else the two overlap by a tenth only, 155 ns per granule and iteration of 2 x 16 columns against
// 69 and 113 apart, and the clock falls to 1.9-2.1 GHz; 32 -> 32 at a million sites is 106 us of that.  Counters there:
// vector unit 52 %, matrix unit 27 % of the time, 1.9 TB/s from beyond L2.
// Against k_conv_split and k_conv_resident, which served these shapes (us, graph replays, room surfaces, 27 taps):
//   sites       1 M        400 k      100 k      24 k       8 k        2 k
//   32 -> 32    262 / 213  105 / 86   44 / 31    24 / 12    18 / 7.6   13 / 7.2
//   16 -> 16    157 / 116  91 / 51    35 / 20    21 / 8.6   21 / 5.6   20 / 5.5
//   48 -> 16    393 / 320  168 / 123  75 / 39    33 / 16    21 / 11    15 / 10
// 8 taps, stride 2, 16 -> 32 from 60 k sites 14 / 5.8; transposed 24 -> 16 onto 20 k sites 8.0 / 4.4; 1x1 16 -> 32 60 k rows 17 / 8.
// Sums of up to 16 channels were computed on fp32 matrix instructions before; against 64 bits (relative 2-norm) 16 -> 16 at
// 20 k sites 2.6e-7 / 6.3e-8, 8 -> 8 1.8e-7 / 6.3e-8, 1x1 8 -> 8 5.7e-8 / 3.3e-8.
template <int NCB, int GW, int DEAL, int OCC, bool PAIR, bool PRE, bool BF16>
__global__ __launch_bounds__(64 * (DEAL > 4 ? DEAL : 4), OCC) void k_conv_wave(
    const int *__restrict__ nbr, const int *__restrict__ rowmap, const unsigned *__restrict__ gmask, int64_t n, int64_t npad,
    const float *__restrict__ in, float *__restrict__ out, const v8s *__restrict__ wp, Epi epi, int n_in, int n_out, int n_slab,
    int ncb, int tiles_per_xcd, int n_tiles, const float *__restrict__ pre_sc, const float *__restrict__ pre_sh, float pre_leak,
    unsigned in_bytes) {
  constexpr int WAVES = DEAL > 4 ? DEAL : 4;
  static_assert(!BF16 || !PAIR, "bf16 operands: whole slabs");
  constexpr int PIECES = BF16 ? 1 : 3;  // of an operand
  static_assert(DEAL == 1 || DEAL == WAVES, "a workgroup is one group of wavefronts that share granules");
  constexpr int PART = DEAL > 1 && NCB > 2 ? NCB : 2;  // KB of LDS per wavefront and granule
  __shared__ v4f turn[WAVES][GW][PART][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int ld_row = lane >> 2, ld_g = lane & 3;
  const int wr_slot = ld_g * 16 + (ld_row ^ (2 * ld_g)), rd_slot = g * 16 + (r16 ^ (2 * g));
  const int tile = tiles_per_xcd ? (blockIdx.x & 7) * tiles_per_xcd + (blockIdx.x >> 3) : blockIdx.x;  // see k_conv_mfma
  if (tile >= n_tiles) return;
  const int64_t pos0 = (DEAL > 1 ? (int64_t)tile : (int64_t)tile * 4 + wave) * (GW * 16);
  if (pos0 >= n) return;  // a wavefront leaves by itself: there are no barriers (DEAL > 1: the whole workgroup)
  const int cb0 = blockIdx.y * NCB;  // first of this wavefront's column blocks, of ncb
  unsigned gm[GW], all = 0u;
#pragma unroll
  for (int q = 0; q < GW; q++) {
    gm[q] = pos0 + 16 * q < n ? __builtin_amdgcn_readfirstlane(gmask[pos0 / 16 + q]) : 0u;
    all |= gm[q];
  }
  const int its = PAIR ? (__popc(all) + 1) / 2 : __popc(all) * n_slab, total = DEAL > 1 ? max(0, (its - wave + DEAL - 1) / DEAL) : its;
  v4f acc[GW][NCB];
#pragma unroll
  for (int q = 0; q < GW; q++)
#pragma unroll
    for (int c = 0; c < NCB; c++) acc[q][c] = (v4f){0.f, 0.f, 0.f, 0.f};

  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(in), 0, (int)in_bytes, 0x00020000);
  const unsigned row_bytes = (unsigned)n_in * 4u;
  const bool tail = n_in % 32 != 0;
  const int last = (int)(n - 1 - pos0);  // positions behind the last one repeat its indices and are left out
  // the taps of `all` in order, lane i the i-th, so that a cursor finds its tap by a lane read however far it moves
  int list = 0;
  if (lane < 32 && ((all >> lane) & 1u)) list = lane + 1;
  list = __builtin_amdgcn_ds_permute(4 * (list ? __popc(all & ((1u << lane) - 1u)) : 63), list) - 1;
  const int n_taps = __popc(all);
  constexpr int TAPS = PAIR ? 2 : 1;  // of an iteration
  // three cursors over the iterations (slab outer, tap inner), each staying on the last one
  struct Cursor {
    int sl, pos, k, k2, left;  // pos: the tap's place in the list; k2 (PAIR): the second tap, -1: none
  };
  auto look = [&](Cursor &c) {
    c.k = __builtin_amdgcn_readlane(list, c.pos);
    if (PAIR) c.k2 = c.pos + 1 < n_taps ? __builtin_amdgcn_readlane(list, c.pos + 1) : -1;
  };
  auto move = [&](Cursor &c, int taps) {
    c.pos += taps;
    if (!PAIR)
      while (c.pos >= n_taps) c.pos -= n_taps, c.sl++;
    look(c);
  };
  auto start = [&](Cursor &c) {
    c = Cursor{0, 0, 0, -1, total};
    if (total > 0) move(c, DEAL > 1 ? wave * TAPS : 0);
  };
  auto advance = [&](Cursor &c) {
    if (c.left <= 1) return;
    c.left--;
    move(c, DEAL * TAPS);
  };
  Cursor at, rows, idx;
  int j[GW][PAIR ? 2 : 1];
  v4f areg[GW][2];
  v8s breg[NCB][PIECES];
  auto issue_indices = [&](const Cursor &c) {
#pragma unroll
    for (int q = 0; q < GW; q++)
#pragma unroll
      for (int h = 0; h < (PAIR ? 2 : 1); h++) {
        const int p = min(16 * q + ld_row, last), k = h && c.k2 >= 0 ? c.k2 : c.k;
        j[q][h] = (nbr + (int64_t)k * npad + pos0)[p];
        if (h && c.k2 < 0) j[q][h] = -1;
      }
  };
  unsigned aok = 0;  // PRE: bit 2q+s: this lane's chunk exists (zero must stay zero)
  v4f psc[2], psh[2];
  auto issue_rows = [&](const Cursor &c) {
    aok = 0;
#pragma unroll
    for (int q = 0; q < GW; q++) {
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const int row = j[q][PAIR ? s : 0], step = PAIR ? 0 : c.sl * 2 + s;  // step: of 16 channels
        const bool past = !BF16 && (PAIR || tail) && step * 16 + 4 * ld_g >= n_in;  // channels past the last
        const bool there = row >= 0 && !past;
        const unsigned off = __umul24((unsigned)row, row_bytes) + 16u * (unsigned)ld_g;
        // (the range check takes the scalar offset from the size: a step past the last channel stays within the one row there may be)
        const unsigned at = BF16 ? (unsigned)step * 64u : min((unsigned)step * 64u, row_bytes);
        areg[q][s] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsrc, there ? off : 0x80000000u, at, 0));
        if (PRE && there) aok |= 1u << (2 * q + s);
      }
    }
    if (PRE) {
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const int ch = (PAIR ? 0 : (c.sl * 2 + s) * 16) + 4 * ld_g;
        psc[s] = *reinterpret_cast<const v4f *>(pre_sc + ch);
        psh[s] = *reinterpret_cast<const v4f *>(pre_sh + ch);
      }
    }
  };
  auto issue_weights = [&](const Cursor &c) {
    if constexpr (PAIR) {  // half an operand from either tap
      const v4s *src = reinterpret_cast<const v4s *>(wp) + lane;
      const v4s *s0 = src + ((int64_t)c.k * (3 * ncb) + cb0) * 64, *s1 = src + ((int64_t)(c.k2 >= 0 ? c.k2 : c.k) * (3 * ncb) + cb0) * 64;
#pragma unroll
      for (int b = 0; b < NCB; b++)
#pragma unroll
        for (int p = 0; p < 3; p++)
          breg[b][p] = __builtin_shufflevector(s0[(p * ncb + b) * 64], s1[(p * ncb + b) * 64], 0, 1, 2, 3, 4, 5, 6, 7);
    } else {
      const v8s *src = wp + (((int64_t)c.k * n_slab + c.sl) * (PIECES * ncb) + cb0) * 64 + lane;
#pragma unroll
      for (int b = 0; b < NCB; b++)
#pragma unroll
        for (int p = 0; p < PIECES; p++) breg[b][p] = src[(p * ncb + b) * 64];
    }
  };
  start(at);
  rows = at;
  idx = at;
  if (total > 0) {
    issue_indices(idx);
    issue_rows(rows);
    issue_weights(rows);
    advance(idx);
    issue_indices(idx);
  }
  for (int it = 0; it < total; it++) {
#pragma unroll
    for (int q = 0; q < GW; q++) {
      if constexpr (BF16) {  // rounded before they turn: half the LDS traffic
        v4f x0 = pre_act<PRE>(areg[q][0], psc[0], psh[0], pre_leak), x1 = pre_act<PRE>(areg[q][1], psc[1], psh[1], pre_leak);
        if (PRE && !((aok >> (2 * q)) & 1u)) x0 = x1 = (v4f){0.f, 0.f, 0.f, 0.f};
        turn[wave][q][0][wr_slot] = __builtin_bit_cast(v4f, to_bf16x8(x0, x1));
        continue;
      }
#pragma unroll
      for (int s = 0; s < 2; s++) {
        v4f v = pre_act<PRE>(areg[q][s], psc[s], psh[s], pre_leak);
        if (PRE && !((aok >> (2 * q + s)) & 1u)) v = (v4f){0.f, 0.f, 0.f, 0.f};
        turn[wave][q][s][wr_slot] = v;
      }
    }
    advance(rows);
    issue_rows(rows);
    advance(idx);
    issue_indices(idx);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < GW; q++) {
      if (!((gm[q] >> at.k) & 1u) && (!PAIR || at.k2 < 0 || !((gm[q] >> at.k2) & 1u))) continue;  // uniform over the wavefront
      if constexpr (BF16) {
        const v8s a = __builtin_bit_cast(v8s, turn[wave][q][0][rd_slot]);
#pragma unroll
        for (int c = 0; c < NCB; c++) {
          // Dealt out, a wavefront's chain is longer than the parts k_conv_rows gave to workgroups on small levels, and the unit does not
          // round its sums to nearest: added up by fp32 adds instead.  Relative 2-norm against 64 bits, k_conv_rows / one chain / so:
          // 1.5 k sites 128 -> 64 9.5e-8 / 1.22e-7 / 8.8e-8, 12 k 128 -> 128 1.58e-7 / 1.59e-7 / 8.6e-8; 1-5 % of the time on small levels
          if constexpr (DEAL > 1) acc[q][c] += mfma_bf16(a, breg[c][0], (v4f){0.f, 0.f, 0.f, 0.f});
          else acc[q][c] = mfma_bf16(a, breg[c][0], acc[q][c]);
        }
      } else {
        const Split8 a = split8(turn[wave][q][0][rd_slot], turn[wave][q][1][rd_slot]);
        v4f t[NCB];
#pragma unroll
        for (int c = 0; c < NCB; c++) t[c] = mfma_bf16(a.h, breg[c][PIECES - 1], (v4f){0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int c = 0; c < NCB; c++) t[c] = mfma_bf16(a.l, breg[c][0], t[c]);
#pragma unroll
        for (int c = 0; c < NCB; c++) t[c] = mfma_bf16(a.m, breg[c][PIECES / 2], t[c]);
#pragma unroll
        for (int c = 0; c < NCB; c++) t[c] = mfma_bf16(a.h, breg[c][PIECES / 2], t[c]);
#pragma unroll
        for (int c = 0; c < NCB; c++) t[c] = mfma_bf16(a.m, breg[c][0], t[c]);
#pragma unroll
        for (int c = 0; c < NCB; c++) t[c] = mfma_bf16(a.h, breg[c][0], t[c]);
#pragma unroll
        for (int c = 0; c < NCB; c++) acc[q][c] += t[c];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    advance(at);
    issue_weights(rows);
  }

  if constexpr (!BF16) {
    float probe = 0.f;  // stays zero while every sum is finite
#pragma unroll
    for (int q = 0; q < GW; q++)
#pragma unroll
      for (int c = 0; c < NCB; c++)
#pragma unroll
        for (int r = 0; r < 4; r++) probe = __builtin_fmaf(acc[q][c][r], 0.f, probe);
    if (__ballot(probe != 0.f) != 0ull) {
      // infinities, NaNs or values too large for pieces: again on the fp32 matrix instructions (see k_conv_split)
#pragma unroll
      for (int q = 0; q < GW; q++)
#pragma unroll
        for (int c = 0; c < NCB; c++) acc[q][c] = (v4f){0.f, 0.f, 0.f, 0.f};
      start(at);
#pragma unroll 1
      for (int it = 0; it < (PAIR ? 2 * total : total); it++) {
        const int k = PAIR && (it & 1) ? at.k2 : at.k, sl = at.sl;
#pragma unroll
        for (int c = 0; c < NCB; c++) {
          if (PAIR && k < 0) break;  // uniform
          float w[8];
          if constexpr (PAIR) {
            const v4s *src = reinterpret_cast<const v4s *>(wp) + ((int64_t)k * (3 * ncb) + cb0 + c) * 64 + lane;
            const v4s wh = src[0], wm = src[ncb * 64], wl = src[2 * ncb * 64];
#pragma unroll
            for (int e = 0; e < 4; e++) w[e] = join_weight(wh[e], wm[e], wl[e]);
          } else {
            const v8s *src = wp + (((int64_t)k * n_slab + sl) * (3 * ncb) + cb0 + c) * 64 + lane;
            const v8s wh = src[0], wm = src[ncb * 64], wl = src[2 * ncb * 64];
#pragma unroll
            for (int e = 0; e < 8; e++) w[e] = join_weight(wh[e], wm[e], wl[e]);
          }
#pragma unroll
          for (int q = 0; q < GW; q++) {
            if (!((gm[q] >> k) & 1u)) continue;  // uniform over the wavefront
            const int *src_j = nbr + (int64_t)k * npad + pos0;
            const int row = 16 * q + r16 <= last ? src_j[16 * q + r16] : -1;
            v4f t = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < (PAIR ? 1 : 2); s++) {
              const int ch = (sl * 2 + s) * 16 + 4 * g;
              const bool there = row >= 0 && ch < n_in;  // n_in is a multiple of four
              v4f x = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                                                  rsrc, there ? (unsigned)row * row_bytes + 4u * (unsigned)ch : 0x80000000u, 0, 0));
              if (PRE) {
                x = pre_act<PRE>(x, *reinterpret_cast<const v4f *>(pre_sc + ch), *reinterpret_cast<const v4f *>(pre_sh + ch), pre_leak);
                if (!there) x = (v4f){0.f, 0.f, 0.f, 0.f};
              }
#pragma unroll
              for (int e = 0; e < 4; e++) t = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], w[4 * s + e], t, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const int p = 16 * q + 4 * g + r;
              acc[q][c][r] += p <= last && src_j[min(p, last)] >= 0 ? t[r] : 0.f;
            }
          }
        }
        if (!PAIR || (it & 1)) advance(at);
      }
    } else {
#pragma unroll
      for (int q = 0; q < GW; q++)
#pragma unroll
        for (int c = 0; c < NCB; c++) acc[q][c] *= SPLIT_UNSCALE;
    }
  }

  // acc[q][c][r] = result for position pos0 + 16*q + 4*g + r, column 16*c + r16
  constexpr int R = DEAL == 1 ? 4 : 1;  // rows per lane and granule that this wavefront stores
  int r0 = 0;
  if constexpr (DEAL > 1) {
    float *sums = reinterpret_cast<float *>(turn);  // [wave][q][c][r][lane]
#pragma unroll
    for (int q = 0; q < GW; q++)
#pragma unroll
      for (int c = 0; c < NCB; c++)
#pragma unroll
        for (int r = 0; r < 4; r++) sums[(((wave * GW + q) * PART + c) * 4 + r) * 64 + lane] = acc[q][c][r];
    __syncthreads();
    if (wave >= 4) return;
    r0 = wave;
#pragma unroll
    for (int q = 0; q < GW; q++)
#pragma unroll
      for (int c = 0; c < NCB; c++) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < DEAL; w++) v += sums[(((w * GW + q) * PART + c) * 4 + wave) * 64 + lane];
        acc[q][c][0] = v;
      }
  }
  const bool post = epi.sc != nullptr;
  float bv[NCB], es[NCB], eh[NCB];
#pragma unroll
  for (int c = 0; c < NCB; c++) {
    const int col = 16 * (cb0 + c) + r16;
    bv[c] = (epi.bias != nullptr && col < n_out) ? epi.bias[col] : 0.0f;
    es[c] = (post && col < n_out) ? epi.sc[col] : 1.0f;
    eh[c] = (post && col < n_out) ? epi.sh[col] : 0.0f;
  }
  const int64_t stride = epi.out_stride ? epi.out_stride : n_out;
  int orow[GW][R];
#pragma unroll
  for (int q = 0; q < GW; q++)
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int p = min(16 * q + 4 * g + r + r0, last);
      orow[q][r] = rowmap ? rowmap[pos0 + p] : (int)pos0 + p;
    }
#pragma unroll
  for (int q = 0; q < GW; q++) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (16 * q + 4 * g + r + r0 > last) continue;
      float *o = out + orow[q][r] * stride + 16 * cb0 + r16;
#pragma unroll
      for (int c = 0; c < NCB; c++) {
        if (16 * (cb0 + c) + r16 >= n_out) continue;
        float v = acc[q][c][r] + bv[c];
        if (epi.out2) epi_second(epi, orow[q][r], 16 * (cb0 + c) + r16, v);
        if (post) v = epi_act(v, es[c], eh[c], epi.leak);
        o[16 * c] = v;
      }
    }
  }
}

template <int NCB, int GW, int DEAL, int OCC, bool PAIR, bool PRE, bool BF16 = false>
static void launch_wave(Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi, int n_in,
                        int n_out, PreArgs pre, hipStream_t s) {
  // what the kernel reads without looking: a slip in the dispatch is an error here, not a read through a null pointer
  if (!t.gmask.p || t.K > 32 || m.fixed_scratch || n_in % 4 || (uintptr_t)in % 16 || m.cur_in_rows * n_in * 4 >= ((int64_t)1 << 31))
    throw Error("internal: this convolution does not fit the kernel chosen for it");
  const int n_slab = (int)ceil_div(n_in, 32);
  const int groups = (int)ceil_div(n_out, 16 * NCB), ncb = groups * NCB;
  const float *wpack;
  if constexpr (BF16) {  // [K][n_slab][ncb][lane], a lane's eight channels of a slab
    const int stride = ncb * 512;
    wpack = packed_weights(m, {6, (int64_t)(uintptr_t)w, t.K, n_in, n_out, ncb}, (size_t)t.K * n_slab * stride / 2, [&](float *dst) {
      launch_pack_weights(w, dst, t.K, n_in, n_out, n_slab, 2, ncb, stride, take_jobs(m), true, s);
    });
  } else {
    wpack = split_weights(m, t.K, w, n_in, n_out, ncb, PAIR, s);
  }
  const int n_tiles = (int)ceil_div(t.n, (DEAL > 1 ? 1 : 4) * GW * 16);
  const int tiles_per_xcd = t.spread ? 0 : (int)ceil_div(n_tiles, 8);
  // (split: workgroups that share a tile's iterations through partial sums in memory, as k_conv_split says it: here never)
  note_kernel(m, BF16 ? "wave-bf16" : "split wave", {{"ncb", NCB}, {"gw", GW}, {"deal", DEAL}, {"pair", PAIR}, {"pre", PRE}, {"split", 1}});
  k_conv_wave<NCB, GW, DEAL, OCC, PAIR, PRE, BF16><<<dim3((unsigned)(tiles_per_xcd ? tiles_per_xcd * 8 : n_tiles), groups), 64 * std::max(4, DEAL), 0, s>>>(
      t.nbr.p, t.rowmap_ptr(), t.gmask.p, t.n, t.npad, in, out, reinterpret_cast<const v8s *>(wpack), epi, n_in, n_out, n_slab,
      ncb, tiles_per_xcd, n_tiles, pre.sc, pre.sh, pre.leak, (unsigned)(m.cur_in_rows * n_in * 4));
  LAUNCH_CHECK();
}

// Taps a position has at most: fine sides of strided tables have few of theirs, as few as coarse and fine rows say (see launch_split).
static int64_t likely_taps(const Table &t, int64_t in_rows) {
  return t.few_tap.p ? 1 : std::min<int64_t>(t.K, ceil_div(t.K * in_rows, std::max<int64_t>(t.n, 1)));
}

// 33 to 48 output planes on small levels: every pair (granules, column group) is a workgroup whose wavefronts deal out the
// iterations, and sums meet in LDS, where k_conv_split writes partial sums for a launch to add up.  Rows are gathered and split
// once per column group and weights read once per workgroup, so that this ends where iterations or granules are many.
// us, k_conv_split with its second launch / here (column blocks, granules, wavefronts of the workgroup chosen):
//   27 taps: 1.2 k sites 48 -> 48 13.0 / 7.9 (2,1,8; three column blocks 9.5), 96 -> 48 15.1 / 10.0, 6 k 48 -> 48 21.4 / 12.9,
//     96 -> 48 22.2 / 17.4, 12 k 48 -> 48 25 / 18, 20 k 29.9 / 24.0 (2,2,4; 30.1 with 2,1,8), 39 k 55 / 41; 300 sites and fewer gain
//     another 1 us from one column block (1,1,8); but 60 sites 100 -> 44 14.2 / 15.8, 140 160 -> 48 15.7 / 18.8, 400 256 -> 48 16.1 / 17.9,
//     9 k 128 -> 48 29.1 / 29.8
//   8 taps, stride 2, onto 25 k sites 32 -> 48 13.8 / 11.5, but onto 8 k 256 -> 48 26.9 / 30.4; one rule per position, onto 3.3 k sites 80 -> 48 8.8 / 4.2, 20 k
//     64 -> 48 9.6 / 6.8, 40 k 12.2 / 10.9; 1x1 1.5 k rows 96 -> 48 6.7 / 3.5, 20 k 8.8 / 6.9
// (64 planes and more would gain as much on levels of a few thousand sites, 1.5 k 64 -> 64 14 / 8; they stay on k_conv_split.)
enum WideTile { NONE, B1G1D8, B2G1D8, B2G2D4 };
static WideTile wide_tile(const Table &t, int64_t in_rows, int n_in, int n_out) {
  if (n_in <= 16 || n_out > 48) return NONE;
  const int64_t n = t.n, slabs = ceil_div(n_in, 32);
  if (t.few_tap.p || t.K == 1) {
    if (n < 5000) return n < 1500 ? B1G1D8 : B2G1D8;
    return n < 25000 || (t.K > 1 && n < 45000 && slabs <= 2) ? B2G2D4 : NONE;
  }
  // long chains on the smallest levels: k_conv_split deals them over more workgroups
  if (slabs >= 4 && n < (slabs == 4 ? 450 : 500) && likely_taps(t, in_rows) > 16) return NONE;
  if (n < 500 && t.K > 9) return slabs <= 5 ? B1G1D8 : NONE;
  if (t.K <= 9) return n < 500 ? B1G1D8 : n < 2500 ? B2G1D8 : n < 25000 && slabs <= 6 ? B2G2D4 : NONE;
  if (n < 10000) return slabs <= (n < 2500 ? 5 : 3) ? B2G1D8 : NONE;
  return n < 40000 && slabs <= 2 ? B2G2D4 : NONE;
}
template <bool PRE>
static void dispatch_wide(Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi, int n_in,
                          int n_out, PreArgs pre, hipStream_t s) {
  switch (wide_tile(t, m.cur_in_rows, n_in, n_out)) {
  case B1G1D8: return launch_wave<1, 1, 8, 4, false, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  case B2G1D8: return launch_wave<2, 1, 8, 4, false, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  case B2G2D4: return launch_wave<2, 2, 4, 4, false, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  case NONE: throw Error("internal: no tile for this convolution");
  }
}
template <int NCB, bool PAIR, bool PRE>
static void dispatch_wave(Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi, int n_in,
                          int n_out, PreArgs pre, hipStream_t s) {
  // the batch norm's coefficients take the registers of one wavefront per SIMD
  constexpr int O1 = PRE && NCB == 2 ? 5 : 6, O2 = PRE && NCB == 2 ? 4 : 5;
  const bool one_rule = t.few_tap.p || t.K == 1;
  // The longer a wavefront's chain, the longer dealing it out pays; many granules per wavefront save weights' traffic where there
  // are enough of them (us: one granule dealt out / two dealt out / two / four):
  //   27 taps 32 -> 32: 8 k sites 7.6 / 9.8 / 25 / 41, 24 k 12.2 / 12.7 / 26 / 42, 100 k 36 / 31 / 36 / 47, 200 k 64 / 52 / 53 / 57,
  //     400 k 120 / 99 / 86 / 90, 1 M 360 / 274 / 230 / 213
  //   9 taps (input gradients only, see conv_wave_serves) 16 -> 16: 12 k 4.7 / 5.4 / 8.4 / 13, 50 k 9.4 / 8.5 / 9.4 / 14, 200 k 31 / 24 / 22 / 26
  //   one rule per position 24 -> 16: 20 k 4.4 / 4.5 / 5.4 / 7.7, 60 k 7.3 / 6.6 / 6.2 / 8.5, 1 M 81 / 55 / 33 / 38
#define WAVE(G, D, O) launch_wave<NCB, G, D, O, PAIR, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s)
  if (t.n < 24000) WAVE(1, 4, O1);
  else if (t.n < (one_rule ? 24000 : t.K <= 9 ? 100000 : 300000)) WAVE(2, 4, O2);
  else if (t.K <= 9 || t.n < 600000) WAVE(2, 1, O2);
  else WAVE(4, 1, 3);
#undef WAVE
}
// bf16 operands (the caller's choice; whole slabs of 32 channels): the same kernel with one instruction and no splitting.  What bounds
// it: what comes from L2, rows and, per wavefront, weights (300 k sites 128 -> 128 269 us: 2.8 GB of read requests, 10.4 TB/s, 1.66 GB of it
// rows; 900 k 32 -> 32 126 us: 1.2 GB of rows, 9.7 TB/s), and on small levels the chain, as above.  us, k_conv_resident,
// k_conv_rows or k_conv_mfma, which keep the rest / here:
//   27 taps: 1 k sites 32 -> 32 18.3 / 4.7, 64 -> 64 12.8 / 6.7, 128 -> 128 18.0 / 10.6; 14 k 32 -> 32 20.0 / 5.8, 64 -> 64 22.6 / 10.6,
//     128 -> 128 36.4 / 27.9, but 256 -> 128 55.9 / 50.7 where 128-row tiles of slabs of 64 (k_conv_rows) take 49.6; 61 k 64 -> 32 47 / 20.5,
//     64 -> 64 38 / 27, but 96 -> 96 60 / 61; 240 k 32 -> 32 60 / 36, 128 -> 64 144 / 134, 128 -> 128 205 / 192; 500 k 32 -> 32 86 / 65,
//     but 64 -> 32 112 / 118; 900 k 32 -> 32 140 / 126
//   8 taps, onto 5 k sites 32 -> 64 13.6 / 4.0, 59 k 13.9 / 12.9, 221 k 32 -> 32 63 / 26; one rule per position, onto 20 k sites
//     64 -> 32 14.0 / 4.1, 900 k 51 / 38, 61 k 96 -> 64 12.8 / 10.9; 1x1 20 k rows 128 -> 64 8.5 / 5.8, 61 k 13.0 / 13.0, 43 k 256 -> 96 19.6 / 24.4
// (Rounding the rows in a pass of its own, so that each rule reads half the bytes, takes longer than it saves: 300 k sites 64 -> 64
// 92 -> 102, 800 k 32 -> 32 99 -> 135.)
// Wide inputs on small levels, where k_conv_rows gives a tile's taps to several workgroups (there / here): 64 sites 256 -> 128 17.8 / 32.5,
// 340 192 -> 64 15.5 / 25.9, 466 160 -> 48 15.2 / 19.0, 700 256 -> 64 18.8 / 26.1, 2.1 k 256 -> 128 28.1 / 34.3, 2.8 k 320 -> 64 31.3 / 37.5; but
// 200 sites 64 -> 64 12.6 / 12.0, 700 96 -> 96 16.9 / 13.4, 1.5 k 128 -> 128 24.7 / 17.0, 6 k 192 -> 32 27.1 / 18.5.  The sites from which on
// this kernel is the faster one, by (many taps) slabs of 32 channels; filter 3 stride 2 from the fine side and eight taps below.
static int64_t bf_from(int64_t taps, int64_t slabs, int n_out) {
  static const int64_t many[3][10] = {{0, 0, 0, 500, 850, 1250, 1800, 2000, 2500, 4500},  // onto up to 32 planes, 64, and more
                                      {0, 0, 0, 520, 850, 1000, 1350, 1500, 4200, 6000},
                                      {0, 0, 0, 400, 600, 700, 1000, 1500, 3000, 3000}};
  if (taps > 16) return many[n_out <= 32 ? 0 : n_out <= 64 ? 1 : 2][std::min<int64_t>(slabs, 9)];
  return taps > 8 ? (slabs >= 8 ? 700 : 0) : taps > 1 && slabs >= 10 ? 250 : 0;
}
enum BfTile { BF_NONE, BF_2_1_4, BF_2_2_4, BF_2_2_1, BF_2_4_1, BF_4_2_4, BF_8_4_1 };  // column blocks, granules, wavefronts that share them
static BfTile bf_tile(const Table &t, int64_t in_rows, int n_in, int n_out) {
  const int64_t n = t.n;
  if (n_in % 32 || n_out > 128) return BF_NONE;
  if (n < bf_from(likely_taps(t, in_rows), n_in / 32, n_out)) return BF_NONE;
  const bool one_rule = t.few_tap.p || t.K == 1, few = one_rule || t.K <= 9;
  if (n_out <= 32) {
    if (n < 20000) return BF_2_1_4;
    if (n < (few ? 100000 : 300000)) return BF_2_2_4;
    if (few) return BF_2_2_1;
    return n_in > 32 ? BF_NONE : n < 700000 ? BF_2_2_1 : BF_2_4_1;
  }
  if (few) {
    const int64_t to = t.K == 1 ? (n_out <= 64 ? 45000 : 28000) : n_out <= 64 ? (one_rule ? 100000 : 70000) : 25000;
    return n < 8000 ? BF_2_1_4 : n < to ? BF_4_2_4 : BF_NONE;
  }
  if (n_out <= 64) return n < 8000 ? BF_2_1_4 : n < 260000 ? BF_4_2_4 : BF_NONE;
  if (n < 3000) return BF_2_1_4;
  if (n_in > 128) return BF_NONE;
  if (n < 8000) return n_out <= 96 ? BF_2_1_4 : BF_4_2_4;
  if (n < 40000) return BF_4_2_4;
  return n_out > 96 && n >= 100000 ? BF_8_4_1 : BF_NONE;
}
template <bool PRE>
static void dispatch_bf(Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi, int n_in,
                        int n_out, PreArgs pre, hipStream_t s) {
#define BF(N, G, D, O) \
  case BF_##N##_##G##_##D: return launch_wave<N, G, D, O, false, PRE, true>(m, t, in, out, w, epi, n_in, n_out, pre, s)
  switch (bf_tile(t, m.cur_in_rows, n_in, n_out)) {
    BF(2, 1, 4, 5);
    BF(2, 2, 4, 4);
    BF(2, 2, 1, 5);
    BF(2, 4, 1, 4);
    BF(4, 2, 4, 4);
    BF(8, 4, 1, 2);
  case BF_NONE: throw Error("internal: no tile for this convolution");
  }
#undef BF
}
bool conv_wave_serves(const Metadata &m, const Table &t, const float *in, int64_t in_rows, int n_in, int n_out, bool gradient) {
  // Forward sums that will be differentiated keep their rounding in k_conv_resident and k_conv_split: with another one values on the edge
  // of a ReLU change sides, and the gradients of a training step over some ten thousand sites differ by up to 9e-3 (2-D: 3.5e-3).  A
  // million-site step takes 1 % longer for it.  So do those over nine taps, whatever the filter's shape, differentiated or not: they are
  // the 3 x 3 filters of 2-D networks, whose time is the host's (1.21 / 1.26 ms for a batch of pen strokes).  The kernels that keep them are slower
  // by themselves (us, there / here, filter 3 x 3 x 1): 4 k sites 16 -> 16 11.7 / 4.6, 32 -> 32 16.4 / 5.3, 48 -> 48 14.0 / 8.2, 100 k 28 / 13, 22 / 19
  // and, bf16 operands, 31 / 14, a million 130 / 73, 141 / 130 and 152 / 101, 64 -> 32 227 / 232.
  if ((t.K == 9 || m.differentiated) && !gradient) return false;
  // The kernel reads granule masks of 32 bits, which tables of more taps do not have (gmask is null there), and keeps its taps in the lanes of
  // half a wavefront; the allocation-free entry has no room for its weights.
  if (m.fixed_scratch || t.K > 32 || !t.gmask.p) return false;
  if (n_in <= 4 || n_in % 4 || (uintptr_t)in % 16 || n_in * 4 >= (1 << 24)) return false;
  if (in_rows <= 0 || in_rows >= (1 << 24) || in_rows * n_in * 4 >= ((int64_t)1 << 31)) return false;
  if (m.bf16) return !gradient && bf_tile(t, in_rows, n_in, n_out) != BF_NONE;  // (these weights are packed from a transposed copy)
  if (n_out > 32) return wide_tile(t, in_rows, n_in, n_out) != NONE;
  // k_conv_resident keeps 20-32 -> up to 16 planes on small levels of few taps and on large ones, where it was faster than k_conv_split, and
  // test_kernel_and_shares_by_size holds the lines.  Here they would be faster still (us, there / here): eight taps onto 1 k to 5 k sites 24 -> 16
  // 11.6-13.1 / 4.3-4.5; 27 taps 32 -> 16 200 k 65 / 41, 300 k 74 / 57, a million 165 / 157, 24 -> 16 300 k 84 / 65, a million 190 / 190.
  if (n_in > 16 && n_in <= 32 && n_out <= 16 && (t.K <= 9 ? t.n < 16000 : t.n >= (n_in > 24 ? 200000 : 300000))) return false;
  // k_conv_split: wide inputs of one rule per position (test_kernel_and_shares_by_size holds them there; transposed 96 -> 32 onto 4 k
  // sites 11.7 us there, 4.6 here, 100 k 20.7 / 15.6, a million 112 / 87, 160 -> 32 13.7 / 5.3, 27.5 / 21.1, 161 / 148), and on the
  // smallest levels chains that it cuts into more parts (500 sites 64 -> 32 11.9 there, 11.1 here, 128 -> 32 13.7 / 18.5, 1.01 k 128 -> 24 17.6 / 21.8,
  // 1.05 k 224 -> 32 21.5 / 33.5, 1.7 k 192 -> 32 22.6 / 29.1, 3.5 k 256 -> 24 37.0 / 43.8, 4.5 k 256 -> 17 35.9 / 41.0, 1.4 k 224 -> 12 23.5 / 29.1; 80 coarse sites of eight taps 256 -> 17 16.5 / 17.4): the
  // sites from which on this kernel is the faster one, by slabs of 32 channels
  static const int64_t many[] = {0, 0, 1000, 1000, 2000, 2500, 3700, 5000, 5500};
  if ((t.few_tap.p && n_in > 64) || (t.K > 9 && t.n < 1000 && n_in > 32)) return false;
  if (likely_taps(t, in_rows) > 16 && t.n < many[std::min<int64_t>(ceil_div(n_in, 32), 8)] * (n_out <= 16 ? 3 : 4) / 4) return false;
  if (t.K > 1 && t.K <= 9 && !t.few_tap.p && t.n < 150 && n_in > 224) return false;
  // k_deconv_few, all weights in LDS (there / here): transposed 32 -> 32 onto 250 k sites 18.0 / 17.4, 500 k 28.0 / 28.5, 1 M 47 / 49, but
  // 64 -> 32 1 M 71 / 64, 60 k 14.4 / 9.6; 1x1 32 -> 32 60 k rows 8.9 / 7.1, 120 k 10.1 / 10.2, 1 M 45 / 58; 64 -> 32 120 k 14.5 / 13.2,
  // 250 k 22.3 / 22.1, 1 M 82 / 93
  if (t.few_tap.p && n_in == 32 && t.n >= 400000) return false;
  if (t.identity_few && (n_in == 32 || n_in == 64) && t.n >= (n_in == 32 ? 100000 : 200000)) return false;
  return true;
}
bool conv_wave_dispatch(bool pre_fused, Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi,
                        int n_in, int n_out, PreArgs pre, hipStream_t s) {
  if (!conv_wave_serves(m, t, in, m.cur_in_rows, n_in, n_out, m.pack_transposed != nullptr)) return false;
  if (m.bf16) {
    pre_fused ? dispatch_bf<true>(m, t, in, out, w, epi, n_in, n_out, pre, s) : dispatch_bf<false>(m, t, in, out, w, epi, n_in, n_out, pre, s);
    return true;
  }
  if (n_out > 32) {
    pre_fused ? dispatch_wide<true>(m, t, in, out, w, epi, n_in, n_out, pre, s) : dispatch_wide<false>(m, t, in, out, w, epi, n_in, n_out, pre, s);
    return true;
  }
  auto run = [&](auto ncb, auto pair) {
    if (pre_fused) dispatch_wave<decltype(ncb)::value, decltype(pair)::value, true>(m, t, in, out, w, epi, n_in, n_out, pre, s);
    else dispatch_wave<decltype(ncb)::value, decltype(pair)::value, false>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  };
  auto by_pair = [&](auto ncb) { n_in <= 16 ? run(ncb, std::true_type()) : run(ncb, std::false_type()); };
  n_out <= 16 ? by_pair(std::integral_constant<int, 1>()) : by_pair(std::integral_constant<int, 2>());
  return true;
}

}  // namespace scn
