// The split-operand MFMA convolution kernel (fp32 results from bf16 matrix instructions) and its
// dispatch; see conv.hip for the family.
#include "conv_common.h"

namespace scn {

// wp[k][slab of 32 channels][piece][column block][lane]: 16 bytes, the lane's eight channels
// (slab*32 + 16*(e/4) + 4*(lane/16) + e%4, e < 8) of column 16*cb + lane%16; zeros outside
// [nIn) x [nOut).
// transposed: `w` is [K][nOut][nIn] (an input gradient's weights as the forward pass has them); mirror: the
// taps in reverse order.  (A transposed copy was a launch per layer of its own, 232 us of the million-site
// U-Net's training step.)
// HALF (up to 16 input channels): wp[k][piece][column block][lane], 8 bytes: the lane's four channels 4*(lane/16) + e, of
// which k_conv_wave puts those of two taps together.
template <bool HALF>
__global__ void k_pack_weights_split(const float *w, void *wp, int K, int n_in, int n_out, int n_slab, int NCB, CoefJobs jobs,
                                     bool transposed, bool mirror) {
  coef_jobs(jobs);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per_slab = (int64_t)NCB * 64;
  if (i >= (int64_t)K * n_slab * per_slab) return;
  const int lane = (int)(i & 63), cb = (int)((i >> 6) % NCB);
  const int64_t ks = i / per_slab;
  const int sl = (int)(ks % n_slab), k = (int)(ks / n_slab);
  const int col = 16 * cb + (lane & 15);
  typedef typename std::conditional<HALF, v4s, v8s>::type Operand;
  Operand h, m, l;
#pragma unroll
  for (int e = 0; e < (HALF ? 4 : 8); e++) {
    const int ch = sl * 32 + 16 * (e >> 2) + 4 * (lane >> 4) + (e & 3);
    float v = 0.0f;
    if (ch < n_in && col < n_out)
      v = transposed ? w[((int64_t)(mirror ? K - 1 - k : k) * n_out + col) * n_in + ch] : w[((int64_t)k * n_in + ch) * n_out + col];
    short ph, pm, pl;
    split_weight(v, ph, pm, pl);
    h[e] = ph, m[e] = pm, l[e] = pl;
  }
  Operand *dst = static_cast<Operand *>(wp) + ks * 3 * per_slab + (int64_t)cb * 64 + lane;
  dst[0] = h;
  dst[per_slab] = m;
  dst[2 * per_slab] = l;
}

// The running convolution's weights in the layout of k_pack_weights_split.
const float *split_weights(Metadata &m, int K, const float *w, int n_in, int n_out, int NCB, bool half, hipStream_t s) {
  const int n_slab = (int)ceil_div(n_in, 32);
  const int64_t threads = (int64_t)K * n_slab * NCB * 64;
  return packed_weights(m, {half ? 5 : 3, (int64_t)(uintptr_t)w, K, n_in, n_out, NCB}, threads * 3 * (half ? 2 : 4), [&](float *dst) {
    auto kern = half ? k_pack_weights_split<true> : k_pack_weights_split<false>;
    kern<<<dim3((unsigned)ceil_div(threads, 256)), 256, 0, s>>>(m.pack_transposed ? m.pack_transposed : w, dst, K, n_in, n_out,
                                                               n_slab, NCB, take_jobs(m), m.pack_transposed != nullptr, m.pack_mirror);
    LAUNCH_CHECK();
  });
}

// A workgroup of 4 wavefronts owns a tile of G = GW*WR granules (16 rows each).  The wavefronts form
// a WR x WC grid: wavefront (wr, wc) keeps, in registers, the accumulators of granules
// [wr*GW, (wr+1)*GW) x column blocks [wc*NCBW, (wc+1)*NCBW).
// Per (slab of 32 input channels, tap) iteration:
//   gathered rows   L2 -> registers, four lanes reading 64 consecutive bytes of a row; split there, once
//                   per row and tile, and written to double-buffered LDS as A operands
//   weights         L2 -> registers: a wavefront's column blocks are its own and the packed layout is
//                   the B operand's lane order
//   MFMAs           CG column blocks at a time over all granules that have the tap; a group's weights
//                   of the next iteration are requested as soon as its MFMAs are issued (no second
//                   set of registers)
// with NB LDS buffers: two and one barrier per iteration, or one and two.  OCC: wavefronts per SIMD that
// the registers are cut for.  An operand slot is moved by twice its lane group so that neither
// the staging writes (lane = row * 4 + chunk) nor the operand reads (lane = chunk * 16 + row) meet in
// a bank.
// Rows or weights that are no finite numbers, or too large for pieces, make the pieces' sums infinite or NaN: a
// wavefront that finds any sum not finite computes its part of the tile again in fp32 (see the end).
template <int NCBW, int WC, int GW, int CG, int NB, int OCC, bool PRE>
__global__ __launch_bounds__(256, OCC) void k_conv_split(
    const int *__restrict__ nbr, const int *__restrict__ rowmap, int K, int64_t n, int64_t npad,
    const float *__restrict__ in, float *__restrict__ out, const v8s *__restrict__ wp, Epi epi, int n_in, int n_out,
    int n_slab, int tiles_per_xcd, int n_tiles, int n_split, float *__restrict__ partial,
    const float *__restrict__ pre_sc, const float *__restrict__ pre_sh, float pre_leak, unsigned in_bytes) {
  constexpr int WR = 4 / WC;
  constexpr int NCB = NCBW * WC;
  constexpr int G = GW * WR;
  constexpr int TM = G * 16;
  constexpr int GPW = G < 4 ? 1 : G / 4;  // granules a wavefront gathers (G < 4: the first G wavefronts)
  constexpr int A_OPS = G * 3 * 64;   // A operands per iteration
  static_assert(G < 4 || G % 4 == 0, "granules must divide over 4 wavefronts");
  extern __shared__ __attribute__((aligned(16))) float lds[];
  v8s *abuf = reinterpret_cast<v8s *>(lds);              // [NB][G][3][64]
  int *jtab = reinterpret_cast<int *>(abuf + NB * A_OPS);  // [G][K][16]
  unsigned *gmask = reinterpret_cast<unsigned *>(jtab + G * K * 16);  // [K] granules having tap k
  int *taplist = reinterpret_cast<int *>(gmask + K);           // [K]
  int *ntaps_p = taplist + K;                                  // [1]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, g = lane >> 4;
  const int ld_row = lane >> 2, ld_g = lane & 3;
  const int wr_slot = ld_g * 16 + (ld_row ^ (2 * ld_g)), rd_slot = g * 16 + (r16 ^ (2 * g));
  const int wr = wave / WC, wc = wave % WC;

  const int tile = tiles_per_xcd ? (blockIdx.x & 7) * tiles_per_xcd + (blockIdx.x >> 3) : blockIdx.x;  // see k_conv_mfma
  if (tile >= n_tiles) return;  // whole workgroup leaves: no barrier is skipped
  const int64_t tbase = (int64_t)tile * TM;
  const int ntaps = tile_setup<256, G, true>(nbr, K, n, npad, tbase, n_split, (int)blockIdx.y, jtab, gmask, taplist, ntaps_p);
  const int total = ntaps * n_slab;
  v4f acc[GW][NCBW];
#pragma unroll
  for (int q = 0; q < GW; q++)
#pragma unroll
    for (int c = 0; c < NCBW; c++) acc[q][c] = (v4f){0.f, 0.f, 0.f, 0.f};

  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(in), 0, (int)in_bytes, 0x00020000);
  const unsigned row_bytes = (unsigned)n_in * 4u;
  const bool tail = n_in % 32 != 0;
  v8s breg[NCBW][3];
  v4f areg[GPW][2];
  v4f psc[2], psh[2];
  unsigned aok = 0;  // bit 2i+s: this lane's chunk of step s of granule i exists (PRE: zero must stay zero)
  unsigned gm_nxt = 0;
  // iteration order: slab outer, tap inner (see k_conv_mfma)
  int nx_ti = 0, nx_sl = 0, nx_k = 0;  // the iteration whose loads are issued next
  auto issue_a = [&]() {
    const int sl = nx_sl;
    gm_nxt = __builtin_amdgcn_readfirstlane(gmask[nx_k]);
    aok = 0;
    if (G < 4 && wave >= G) return;
#pragma unroll
    for (int i = 0; i < GPW; i++) {
      const int j = jtab[((wave * GPW + i) * K + nx_k) * 16 + ld_row];
      const unsigned voff = j >= 0 ? __umul24((unsigned)j, row_bytes) + 16u * (unsigned)ld_g : 0x80000000u;
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const bool past = tail && (sl * 2 + s) * 16 + 4 * ld_g >= n_in;  // channels past the last
        // (the range check takes the scalar offset from the size: a step past the last channel stays within the one row there may be)
        const unsigned at = min((unsigned)(sl * 2 + s) * 64u, row_bytes);
        areg[i][s] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsrc, past ? 0x80000000u : voff, at, 0));
        if (PRE && j >= 0 && !past) aok |= 1u << (2 * i + s);
      }
    }
    if (PRE) {
#pragma unroll
      for (int s = 0; s < 2; s++) {
        psc[s] = *reinterpret_cast<const v4f *>(pre_sc + (sl * 2 + s) * 16 + 4 * ld_g);
        psh[s] = *reinterpret_cast<const v4f *>(pre_sh + (sl * 2 + s) * 16 + 4 * ld_g);
      }
    }
  };
  auto issue_b = [&](int c) {
    const v8s *src = wp + ((int64_t)nx_k * n_slab + nx_sl) * (3 * NCB * 64) + (wc * NCBW + c) * 64 + lane;
#pragma unroll
    for (int p = 0; p < 3; p++) breg[c][p] = src[p * NCB * 64];
  };
  auto advance = [&]() {  // stays on the last iteration
    if (nx_sl * ntaps + nx_ti + 1 >= total) return;
    if (++nx_ti == ntaps) nx_ti = 0, nx_sl++;
    nx_k = __builtin_amdgcn_readfirstlane(taplist[nx_ti]);
  };

  if (total > 0) {
    nx_k = __builtin_amdgcn_readfirstlane(taplist[0]);
    issue_a();
#pragma unroll
    for (int c = 0; c < NCBW; c++) issue_b(c);
  }
  for (int it = 0; it < total; it++) {
    v8s *ab = abuf + (NB == 2 ? (it & 1) * A_OPS : 0);
    if (NB == 1 && it > 0) __syncthreads();  // every wavefront has read the rows of it-1
#pragma unroll
    for (int i = 0; i < GPW; i++) {
      const int gr = wave * GPW + i;
      if (G < 4 && wave >= G) break;
      v4f v[2];
#pragma unroll
      for (int s = 0; s < 2; s++) {
        v[s] = pre_act<PRE>(areg[i][s], psc[s], psh[s], pre_leak);
        if (PRE && !((aok >> (2 * i + s)) & 1u)) v[s] = (v4f){0.f, 0.f, 0.f, 0.f};
      }
      const Split8 p = split8(v[0], v[1]);
      ab[(gr * 3 + 0) * 64 + wr_slot] = p.h;
      ab[(gr * 3 + 1) * 64 + wr_slot] = p.m;
      ab[(gr * 3 + 2) * 64 + wr_slot] = p.l;
    }
    const unsigned gm = gm_nxt;
    // After this barrier the rows of `it` are visible, and every wavefront has finished the MFMAs of
    // it-1, so the other buffer may be overwritten at the top of it+1.
    __syncthreads();
    advance();
    issue_a();
#pragma unroll
    for (int c0 = 0; c0 < NCBW; c0 += CG) {
#pragma unroll
      for (int q = 0; q < GW; q++) {
        const int gr = wr * GW + q;
        if (!((gm >> gr) & 1u)) continue;  // uniform over the wavefront
        const v8s ah = ab[(gr * 3 + 0) * 64 + rd_slot], am = ab[(gr * 3 + 1) * 64 + rd_slot],
                  al = ab[(gr * 3 + 2) * 64 + rd_slot];
        v4f t[CG];
#pragma unroll
        for (int c = 0; c < CG; c++) t[c] = mfma_bf16(ah, breg[c0 + c][2], (v4f){0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int c = 0; c < CG; c++) t[c] = mfma_bf16(al, breg[c0 + c][0], t[c]);
#pragma unroll
        for (int c = 0; c < CG; c++) t[c] = mfma_bf16(am, breg[c0 + c][1], t[c]);
#pragma unroll
        for (int c = 0; c < CG; c++) t[c] = mfma_bf16(ah, breg[c0 + c][1], t[c]);
#pragma unroll
        for (int c = 0; c < CG; c++) t[c] = mfma_bf16(am, breg[c0 + c][0], t[c]);
#pragma unroll
        for (int c = 0; c < CG; c++) t[c] = mfma_bf16(ah, breg[c0 + c][0], t[c]);
#pragma unroll
        for (int c = 0; c < CG; c++) acc[q][c0 + c] += t[c];
      }
#pragma unroll
      for (int c = 0; c < CG; c++) issue_b(c0 + c);
    }
  }

  float probe = 0.f;  // stays zero while every sum is finite
#pragma unroll
  for (int q = 0; q < GW; q++)
#pragma unroll
    for (int c = 0; c < NCBW; c++)
#pragma unroll
      for (int r = 0; r < 4; r++) probe = __builtin_fmaf(acc[q][c][r], 0.f, probe);
  if (__ballot(probe != 0.f) != 0ull) {
    // Infinities, NaNs or values too large for pieces: the wavefront's part of the tile again on the fp32
    // matrix instructions, rows as they are and weights put back together from their pieces (the packed
    // layout is the operand order of these instructions too: element e of step s is the lane's channel of one
    // of them).  A row that does not have the tap is left out of the sum, not multiplied as zeros: its
    // weights may be infinite.  Where every tile has to, a pass takes 1.5 (20 k sites 32 -> 32), 2 (64 -> 64), 3
    // (128 -> 128) or 4 to 5 times (256 -> 256) an ordinary one; a loop over single values took 27 to 216 times.
#pragma unroll
    for (int q = 0; q < GW; q++)
#pragma unroll
      for (int c = 0; c < NCBW; c++) acc[q][c] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int it = 0; it < total; it++) {
      const int ti = it / n_slab, sl = it - ti * n_slab;
      const int k = __builtin_amdgcn_readfirstlane(taplist[ti]);
      const unsigned gm = __builtin_amdgcn_readfirstlane(gmask[k]);
#pragma unroll
      for (int c = 0; c < NCBW; c++) {
        const v8s *src = wp + ((int64_t)k * n_slab + sl) * (3 * NCB * 64) + (wc * NCBW + c) * 64 + lane;
        const v8s wh = src[0], wm = src[NCB * 64], wl = src[2 * NCB * 64];
        float w[8];
#pragma unroll
        for (int e = 0; e < 8; e++) w[e] = join_weight(wh[e], wm[e], wl[e]);
#pragma unroll
        for (int q = 0; q < GW; q++) {
          const int gr = wr * GW + q;
          if (!((gm >> gr) & 1u)) continue;  // uniform over the wavefront
          const int *rows = jtab + (gr * K + k) * 16;
          const int j = rows[r16];
          v4f t = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int s = 0; s < 2; s++) {
            const int ch = (sl * 2 + s) * 16 + 4 * g;
            const bool there = j >= 0 && ch < n_in;  // n_in is a multiple of four
            v4f x = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                                                rsrc, there ? (unsigned)j * row_bytes + 4u * (unsigned)ch : 0x80000000u, 0, 0));
            if (PRE) {
              x = pre_act<PRE>(x, *reinterpret_cast<const v4f *>(pre_sc + ch), *reinterpret_cast<const v4f *>(pre_sh + ch), pre_leak);
              if (!there) x = (v4f){0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int e = 0; e < 4; e++) t = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], w[4 * s + e], t, 0, 0, 0);
          }
#pragma unroll
          for (int r = 0; r < 4; r++) acc[q][c][r] += rows[4 * g + r] >= 0 ? t[r] : 0.f;
        }
      }
    }
  } else {
#pragma unroll
    for (int q = 0; q < GW; q++)
#pragma unroll
      for (int c = 0; c < NCBW; c++) acc[q][c] *= SPLIT_UNSCALE;
  }

  // acc[q][c][r] = result for position tbase + 16*(wr*GW+q) + 4*g + r, column 16*(wc*NCBW+c) + r16
  if (partial) {  // [n_split][n_tiles * TM][NCB * 16]
    float *pt = partial + ((int64_t)blockIdx.y * n_tiles * TM + tbase) * (NCB * 16);
#pragma unroll
    for (int q = 0; q < GW; q++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int p = (wr * GW + q) * 16 + 4 * g + r;
        if (tbase + p >= n) continue;
#pragma unroll
        for (int c = 0; c < NCBW; c++) pt[(int64_t)p * (NCB * 16) + 16 * (wc * NCBW + c) + r16] = acc[q][c][r];
      }
    return;
  }
  const bool post = epi.sc != nullptr;
  float bv[NCBW], es[NCBW], eh[NCBW];
#pragma unroll
  for (int c = 0; c < NCBW; c++) {
    const int col = 16 * (wc * NCBW + c) + r16;
    bv[c] = (epi.bias != nullptr && col < n_out) ? epi.bias[col] : 0.0f;
    es[c] = (post && col < n_out) ? epi.sc[col] : 1.0f;
    eh[c] = (post && col < n_out) ? epi.sh[col] : 0.0f;
  }
#pragma unroll
  for (int q = 0; q < GW; q++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int64_t pos = tbase + (wr * GW + q) * 16 + 4 * g + r;
      if (pos >= n) continue;
      const int64_t row = rowmap ? rowmap[pos] : pos;
#pragma unroll
      for (int c = 0; c < NCBW; c++) {
        const int col = 16 * (wc * NCBW + c) + r16;
        if (col >= n_out) continue;
        float v = acc[q][c][r] + bv[c];
        if (epi.out2) epi_second(epi, row, col, v);
        if (post) v = epi_act(v, es[c], eh[c], epi.leak);
        out[row * (epi.out_stride ? epi.out_stride : n_out) + col] = v;
      }
    }
  }
}

template <int NCBW, int WC, int GW, int CG, int NB, int OCC, bool PRE>
static bool launch_split(Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi, int n_in,
                         int n_out, PreArgs pre, hipStream_t s) {
  constexpr int WR = 4 / WC, NCB = NCBW * WC, G = GW * WR;
  const size_t lds_bytes = (size_t)NB * G * 3 * 64 * 16 + ((size_t)G * t.K * 16 + 2 * t.K + 4) * sizeof(int);
  if (lds_bytes > 160 * 1024) return false;
  const int n_slab = (int)ceil_div(n_in, 32);
  const float *wpack = split_weights(m, t.K, w, n_in, n_out, NCB, false, s);
  constexpr int CUT = !PRE || OCC == 4 ? OCC : OCC == 5 ? 3 : 2;  // the batch norm's coefficients take 16 registers more
  auto kern = k_conv_split<NCBW, WC, GW, CG, NB, CUT, PRE>;
  static bool attr_set = false;
  if (!attr_set) {
    HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  160 * 1024));
    attr_set = true;
  }
  const int n_tiles = (int)ceil_div(t.n, G * 16);
  const int tiles_per_xcd = t.spread ? 0 : (int)ceil_div(n_tiles, 8);  // 0: tile = workgroup index
  // Few tiles: the taps of a tile dealt over several workgroups, four of 64 rows (or two of 128) per CU in
  // all, and a launch adds the parts up.  (Two and only below 256 tiles, as the fp32 kernels have it, is slower: 20 k
  // sites 64 -> 64 48 -> 29 us, 30 k 128 -> 128 126 -> 91, 14 k 256 -> 128 116 -> 91; six per CU the same within
  // 5 % either way.)  `chain`: iterations of a tile.  The fine side of a transposed table has K * (coarse sites / fine
  // sites) rules per position at most, and its positions are ordered by tap or pattern, so that from some 50 tiles on a
  // tile has about as few taps.  Not dealt out, in us (graph replays):
  //   one rule per position and tiles that mostly have one tap: 5 k fine sites 64 -> 256 30.2 dealt out, 24.4 not;
  //     20 k 64 -> 64 23.1 / 13.8, 96 -> 96 28.0 / 18.9; but 300 sites 96 -> 96 11.8 / 17
  //   chains of up to 12 where the level itself has the workgroups: 20 k fine sites, filter 3 stride 2, 32 -> 64 23.0 / 18.9;
  //     eight iterations, 1 k coarse sites 32 -> 64 10.0 / 13.3, 5 k 11 / 16, but 10 k 21.4 / 15.8; up to 32 output planes gain
  //     less on the device (nine taps 24 -> 32 16 / 11) than a second launch costs a host that issues them one by one
  // Parts of three iterations and more keep the partial sums and the time to add them small: 2 k sites 32 -> 64 20.4 us
  // with parts of one, 15.1; 64 -> 64 21.9 / 19.2; 128-row tiles and the shortest chains are better off without (1 k sites
  // 64 -> 32 15.5 / 16.0, 1.2 k coarse sites 32 -> 64 10.0 / 11.4).
  const int64_t taps = t.n < 768 * G ? t.K : std::min<int64_t>(t.K, ceil_div(t.K * m.cur_in_rows, t.n));
  const int64_t chain = taps * n_slab;
  const bool one_rule = t.few_tap.p && t.n >= 1024 * G;
  const int part = NCB <= 2 || (chain <= 24 && t.n < 2500) ? 1 : 3;
  int n_split = 1;
  if (n_tiles < 512 && !one_rule && (chain > 12 || (chain > 7 && t.n < 6000 && NCB > 2)))
    n_split = (int)std::min<int64_t>({t.K, ceil_div(t.n < 3000 ? 3072 : 4096, (int64_t)n_tiles * G), ceil_div(chain, part)});
  const int64_t split_stride = (int64_t)n_tiles * G * 16 * NCB * 16;
  float *partial = scratch_partial(m, n_split, split_stride);
  note_kernel(m, "split", {{"ncbw", NCBW}, {"wc", WC}, {"gw", GW}, {"pre", PRE}, {"split", n_split}});
  kern<<<dim3((unsigned)(tiles_per_xcd ? tiles_per_xcd * 8 : n_tiles), n_split), 256, lds_bytes, s>>>(
      t.nbr.p, t.rowmap_ptr(), t.K, t.n, t.npad, in, out, reinterpret_cast<const v8s *>(wpack), epi, n_in, n_out, n_slab,
      tiles_per_xcd, n_tiles, n_split, partial, pre.sc, pre.sh, pre.leak, (unsigned)(m.cur_in_rows * n_in * 4));
  LAUNCH_CHECK();
  if (n_split > 1) launch_conv_reduce(partial, n_split, split_stride, NCB * 16, t.rowmap_ptr(), t.n, epi, out, n_out, s);
  return true;
}

// The tile by width and size of the level (us, eval layers on room surfaces; "was": the fp32 kernel
// that served the shape before).
//   widths of up to 128 planes, from 300 k sites on: 128-row tiles with one LDS buffer (two
//   barriers an iteration, but three to five workgroups per CU instead of two): a million sites
//     32 -> 32 257 -> 234, 64 -> 32 464 -> 393, 64 -> 64 838 -> 558 (64-row tiles 599), 96 -> 96 1744 -> 1134
//     (1229), 128 -> 128 2928 -> 1742 (1759)
//   below, 64-row tiles with two buffers, twice the workgroups for a level of a few waves of them:
//     247 k 128 -> 64 415 -> 293 (128-row 307), 200 k 48 -> 64 207 -> 133 (144), 61 k 96 -> 96 171 -> 110 (139),
//     3 k 128 -> 128 37 -> 27 (35); 32 output planes keep 128-row tiles, which lose nothing there
//   below 1024 sites, 32-row tiles beyond 32 planes: a launch is as long as one workgroup's chain; 300
//     sites 64 -> 64 10.6 (64-row tiles 11.0, was 10.8), 768 192 -> 192 22.8 (25.7, was 29.6), 384 -> 192 32.4
//     (36.3, was 46.1); 152 sites 224 -> 224 21.4 (23.3, was 19.1); at 3.3 k 320 -> 160 68 against 57
//   and up to 24 k where a tile has only a few iterations (1x1 convolutions, the fine side of filter = stride tables, eight
//     or nine taps of 32 planes), for the same reason: 64 -> 256 1x1 5 k rows 19.8 -> 12.1, 20 k 23.9 -> 16.8; transposed 96 -> 96
//     10 k sites 16.8 -> 14.5; 40 k one way or the other
//   wider: 64-row tiles, three wavefronts per SIMD: a million sites 256 -> 256 11561 -> 6851 (128-row
//     tiles, two wavefronts 6856), 100 k 1553 -> 830 (880); 300 k 192 -> 192 2336 -> 1276 (1359), 60 k
//     160 -> 160 507 -> 290 (304), 3.3 k 160 -> 160 42 -> 37
// At 1240 TFLOP/s of bf16 products the widest layers run at what a large bf16 matrix product of the
// vendor's library reaches on this card; the narrow ones are bound by operand traffic (a 32 x 32 wavefront
// tile reads 12 KB of operands for 384 matrix cycles).
template <bool PRE>
static bool dispatch_split(Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi, int n_in,
                           int n_out, PreArgs pre, hipStream_t s) {
  const int ncb = (int)ceil_div(n_out, 16);
  const bool large = t.n >= 300000;
  const bool short_chain = t.few_tap.p || t.K * ceil_div(n_in, 32) <= 9;
  if (t.n < 1024 || (t.n < 24000 && short_chain)) {
    if (ncb > 2 && ncb <= 4) return launch_split<2, 2, 1, 2, 2, 2, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
    if (ncb > 4 && ncb <= 6) return launch_split<3, 2, 1, 3, 2, 2, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
    if (ncb > 6 && ncb <= 8) return launch_split<2, 4, 2, 2, 2, 2, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
    if (ncb > 8 && ncb <= 10) return launch_split<5, 2, 1, 5, 2, 2, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
    if (ncb > 10 && ncb <= 12) return launch_split<3, 4, 2, 3, 2, 2, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
    if (ncb > 12 && ncb <= 14) return launch_split<7, 2, 1, 7, 2, 2, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
    if (ncb > 14 && ncb <= 16) return launch_split<4, 4, 2, 4, 2, 2, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  }
  if (ncb <= 2) return launch_split<2, 1, 2, 2, 1, 5, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  if (ncb <= 4)
    return large ? launch_split<2, 2, 4, 2, 1, 3, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s)
                 : launch_split<2, 2, 2, 2, 2, 2, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  if (ncb <= 6)
    return large ? launch_split<3, 2, 4, 3, 1, 3, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s)
                 : launch_split<3, 2, 2, 3, 2, 2, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  if (ncb <= 8)
    return large ? launch_split<2, 4, 8, 2, 1, 3, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s)
                 : launch_split<2, 4, 4, 2, 2, 4, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  if (ncb <= 10) return launch_split<5, 2, 2, 5, 2, 2, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  if (ncb <= 12) return launch_split<3, 4, 4, 3, 2, 3, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  if (ncb <= 14) return launch_split<7, 2, 2, 7, 2, 2, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  if (ncb <= 16) return launch_split<4, 4, 4, 4, 2, 3, PRE>(m, t, in, out, w, epi, n_in, n_out, pre, s);
  return false;
}

// What the fp32 kernels keep (us):
//   inputs of up to 16 planes: half of a 32-channel slab would be empty (a million sites 16 -> 16 146 there, 193
//     here; 24 -> 24 265 there, 243 here, and 67 / 21 at 20 k sites)
//   up to 32 -> 16 planes at large levels, where half of the columns here would be empty too and staging all weights per
//     workgroup does not show any more: 32 -> 16 a million sites 164 there, 222 here, 400 k 83 / 98, 200 k 62 / 64, 150 k
//     63 / 55; 20 -> 16 a million 187 / 225, 300 k 83 / 83; eight taps the other way round (a million fine sites 70 / 36)
//   up to nine taps of up to 32 planes onto up to 16 on small levels (24 -> 16, 8 taps: 250 coarse sites 13.4 / 14.9, 10 k 15.5 /
//     16.1, 20 k 17.4 / 16.3)
//   more than 64 taps onto up to 32 planes: 128 rows of so many neighbour indices leave one workgroup per CU (5^3,
//     100 k sites 32 -> 32 353 / 443, 64 -> 32 675 / 831, 1 k 25 / 34; 49 taps 50 k 32 -> 32 73 / 76, 24 -> 32 91 / 76)
//   the allocation-free entry point: its fixed array holds fp32 weights, not half as many again
bool conv_split_serves(const Metadata &m, const Table &t, const float *in, int64_t in_rows, int n_in, int n_out) {
  if (m.bf16 || m.fixed_scratch) return false;
  if (n_in <= 16 || n_in % 4 || (uintptr_t)in % 16 || t.K > 1024 || n_in * 4 >= (1 << 24)) return false;
  if (n_out <= 16 && n_in <= 32 && (t.K <= 9 ? t.n < 16000 : t.n >= (n_in > 24 ? 200000 : 300000)) &&
      resident_fits(m, t, n_in, n_out, false))
    return false;
  if (n_out <= 32 && t.K > 64) return false;
  return in_rows > 0 && in_rows < (1 << 24) && in_rows * n_in * 4 < ((int64_t)1 << 31);
}
bool conv_split_dispatch(bool pre_fused, Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi,
                         int n_in, int n_out, PreArgs pre, hipStream_t s) {
  if (!conv_split_serves(m, t, in, m.cur_in_rows, n_in, n_out)) return false;
  return pre_fused ? dispatch_split<true>(m, t, in, out, w, epi, n_in, n_out, pre, s)
                   : dispatch_split<false>(m, t, in, out, w, epi, n_in, n_out, pre, s);
}

}  // namespace scn
