// Weight gradients of wide layers, fp32 operands as three bf16 pieces; see backward.hip for the family.
#include "conv_common.h"

namespace scn {

constexpr int DS_BLOCK = 8;  // granules of 16 positions that are dealt together

// dW[k][c][o] = sum over positions t with nbr[k][t] >= 0 of a[nbr[k][t]][c] * b[row(t)][o].
// A workgroup owns tap k, a tile of 32 NA x 32 NB channels and a share of the positions; its 2 x 2
// wavefronts own 16 NA x 16 NB channels each.  Per iteration it takes 2 KS granules that have the tap:
//   staging  a thread gathers four consecutive channels of eight positions (four of either granule of a
//            pair: 16-byte loads, an iteration ahead), splits the 32 values (split8) and writes four
//            operands of each piece: the MFMA contracts over 32 positions, an operand is one channel
//            at eight of them
//   MFMAs    16x16x32, six per pair of operands and 32 positions, summed from zero and added in fp32
// Channel 4 q + i of a side (quad q of 8 N quads) is row L % 16 of operand block L / 16 with L = 8 N i + q:
// consecutive threads stage consecutive quads, so that their 16-byte writes are consecutive too.
// What bounds it: the vector instructions of the splitting next to the MFMAs (a value is split once per
// workgroup; once per wavefront, without LDS, took 4.3 ms where this takes 2.5), and the gathers' latency at
// two workgroups per CU.  Against the fp32 kernel (us, kernel alone): a million sites 128 x 128 4600 -> 2674,
// 64 x 64 1113 -> 875; 247 k 128 x 64 564 -> 431; 61 k 192 x 96 474 -> 274, 96 x 96 198 -> 152; 14 k 128 x 128 92 -> 75;
// 3.3 k 160 x 160 85 -> 65.  All taps have the same shares, so that no rule counts are fetched from the device.
template <int NA, int NB>
__global__ __launch_bounds__(256, 2) void k_conv_dw_split(
    const int *__restrict__ nbr, const int *__restrict__ rowmap, const unsigned *__restrict__ gmask, int K, int64_t n,
    int64_t npad, const float *__restrict__ a, int n_a, unsigned a_bytes, const float *__restrict__ b, int n_b,
    unsigned b_bytes, int shares, int in_turns, float *__restrict__ partial) {
  constexpr int KS = 8 / (NA + NB);  // pairs of granules per iteration
  constexpr int STEP_T = 32 * (NA + NB);                     // threads that stage a pair
  constexpr int BLK = 2 * (NA + NB);                         // operand blocks of a pair (a's first)
  __shared__ v8s ops[KS][3][BLK][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, g = lane >> 4;
  const int mt_b = (n_b + 32 * NB - 1) / (32 * NB), mt = (n_a + 32 * NA - 1) / (32 * NA) * mt_b;
  // Workgroups are dealt round-robin to the 8 XCDs: an XCD takes every eighth share, and all taps and
  // tiles of a share one after the other, so that the rows of its positions come from one L2.
  const int local = blockIdx.x >> 3, per_share = K * mt;
  const int share = (blockIdx.x & 7) + 8 * (local / per_share);
  if (share >= shares) return;  // uniform over the workgroup
  const int k = local % per_share / mt, tile = local % mt;
  const int ca0 = tile / mt_b * 32 * NA, cb0 = tile % mt_b * 32 * NB;
  const int wr = wave >> 1, wc = wave & 1;
  // staging role
  const int step = threadIdx.x / STEP_T, u = threadIdx.x % STEP_T;
  const bool stages = step < KS, side_a = u < 32 * NA;
  const int quads = side_a ? 8 * NA : 8 * NB, v = side_a ? u : u - 32 * NA;
  const int sq = v % quads, sg = v / quads;
  const int sc = (side_a ? ca0 : cb0) + 4 * sq;  // first of the thread's four channels
  const bool has_channels = stages && sc < (side_a ? n_a : n_b);
  const unsigned nowhere = 0x80000000u;  // offsets from here on read zeros
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a), 0, (int)a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(b), 0, (int)b_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t nbr_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int *>(nbr), 0, (int)((unsigned)K * (unsigned)npad * 4u), 0x00020000);
  const __amdgpu_buffer_rsrc_t map_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int *>(rowmap ? rowmap : nbr), 0, (int)((unsigned)npad * 4u), 0x00020000);
  const int n_granules = (int)((n + 15) >> 4), n32 = (int)n;
  // The share's granules with the tap, in ascending order: blocks first, first + stride, ... below end.  A
  // wavefront (all four alike) looks at eight blocks at a time, a lane per granule (one load, a ballot),
  // and has the masks of the next eight on their way.
  const int n_blocks = (n_granules + DS_BLOCK - 1) / DS_BLOCK;
  const int first = in_turns ? share : (int)((int64_t)share * n_blocks / shares);
  const int end = in_turns ? n_blocks : (int)((int64_t)(share + 1) * n_blocks / shares);
  const int stride = in_turns ? shares : 1;
  const __amdgpu_buffer_rsrc_t gm_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<unsigned *>(gmask ? gmask : reinterpret_cast<const unsigned *>(nbr)), 0, (int)((unsigned)n_granules * 4u), 0x00020000);
  int look = 0;           // blocks (of this share) in front of the look that `found` is of
  uint64_t found = 0ull;  // its granules with the tap still to come
  unsigned ahead = 0u;    // this lane's mask of the next look
  int ahead_at = 0;
  const int shift = gmask ? k : 0;
  auto request = [&](int at) {
    const int blk = first + (at + (lane >> 3)) * stride, gi = blk * DS_BLOCK + (lane & 7);
    const bool in = blk < end && gi < n_granules;
    ahead_at = at;
    ahead = in ? 1u : 0u;
    if (gmask) ahead = __builtin_amdgcn_raw_buffer_load_b32(gm_rsrc, in ? (unsigned)gi * 4u : nowhere, 0, 0);
  };
  auto next_granule = [&]() {  // n_granules: none
    while (found == 0ull) {
      if (first + ahead_at * stride >= end) return n_granules;
      look = ahead_at;
      found = __ballot((ahead >> shift) & 1u);
      request(look + 8);
    }
    const int bit = __builtin_ctzll(found);
    found &= found - 1ull;
    return (first + (look + (bit >> 3)) * stride) * DS_BLOCK + (bit & 7);
  };

  v4f acc[NA][NB];
#pragma unroll
  for (int i = 0; i < NA; i++)
#pragma unroll
    for (int j = 0; j < NB; j++) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  int gq[2 * KS];         // granules whose indices are in `idx`
  int4 idx[2];            // rows of this thread's side at its four positions of either granule
  v4f raw[2][4];          // four channels of those rows
  auto load_indices = [&](int gi, int4 &j) {
    const int t = gi * 16 + 4 * sg;
    const unsigned toff = gi < n_granules ? (unsigned)t * 4u : nowhere;
    j = make_int4(t, t + 1, t + 2, t + 3);
    if (side_a)
      j = __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(nbr_rsrc, toff, (unsigned)k * (unsigned)npad * 4u, 0));
    else if (rowmap)
      j = __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(map_rsrc, toff, 0, 0));
  };
  auto seek_and_index = [&]() {
#pragma unroll
    for (int q = 0; q < 2 * KS; q++) gq[q] = next_granule();
    int g0 = gq[0], g1 = gq[1];
#pragma unroll
    for (int s = 1; s < KS; s++)
      if (step == s) g0 = gq[2 * s], g1 = gq[2 * s + 1];
    load_indices(g0, idx[0]);
    load_indices(g1, idx[1]);
  };
  auto load_rows = [&]() {
    int g0 = gq[0], g1 = gq[1];
#pragma unroll
    for (int s = 1; s < KS; s++)
      if (step == s) g0 = gq[2 * s], g1 = gq[2 * s + 1];
    unsigned off[2][4];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int j[4] = {idx[h].x, idx[h].y, idx[h].z, idx[h].w}, gi = h ? g1 : g0;
#pragma unroll
      for (int x = 0; x < 4; x++) {
        const bool live = has_channels && gi < n_granules && gi * 16 + 4 * sg + x < n32 && j[x] >= 0;
        off[h][x] = live ? ((unsigned)j[x] * (unsigned)(side_a ? n_a : n_b) + (unsigned)sc) * 4u : nowhere;
      }
    }
    if (side_a) {
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int x = 0; x < 4; x++)
          raw[h][x] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, off[h][x], 0, 0));
    } else {
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int x = 0; x < 4; x++)
          raw[h][x] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, off[h][x], 0, 0));
    }
  };
  request(0);
  seek_and_index();
  bool more = gq[0] < n_granules;  // uniform over the workgroup
  load_rows();
  int used[2 * KS];
#pragma unroll
  for (int q = 0; q < 2 * KS; q++) used[q] = gq[q];
  seek_and_index();
  while (more) {
    if (stages) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const Split8 p = split8((v4f){raw[0][0][i], raw[0][1][i], raw[0][2][i], raw[0][3][i]},
                                (v4f){raw[1][0][i], raw[1][1][i], raw[1][2][i], raw[1][3][i]});
        const int L = i * quads + sq, blk = (side_a ? 0 : 2 * NA) + (L >> 4), slot = sg * 16 + (L & 15);
        ops[step][0][blk][slot] = p.h;
        ops[step][1][blk][slot] = p.m;
        ops[step][2][blk][slot] = p.l;
      }
    }
    __syncthreads();  // the operands are in LDS
    load_rows();
    int cur[2 * KS];
#pragma unroll
    for (int q = 0; q < 2 * KS; q++) cur[q] = used[q], used[q] = gq[q];
    more = gq[0] < n_granules;
    seek_and_index();
#pragma unroll
    for (int s = 0; s < KS; s++) {
      if (s > 0 && cur[2 * s] >= n_granules) continue;  // uniform
      v8s pb[NB][3];
#pragma unroll
      for (int j = 0; j < NB; j++)
#pragma unroll
        for (int p = 0; p < 3; p++) pb[j][p] = ops[s][p][2 * NA + wc * NB + j][lane];
#pragma unroll
      for (int i = 0; i < NA; i++) {
        const v8s ah = ops[s][0][wr * NA + i][lane], am = ops[s][1][wr * NA + i][lane], al = ops[s][2][wr * NA + i][lane];
        v4f t[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) t[j] = mfma_bf16(ah, pb[j][2], (v4f){0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int j = 0; j < NB; j++) t[j] = mfma_bf16(al, pb[j][0], t[j]);
#pragma unroll
        for (int j = 0; j < NB; j++) t[j] = mfma_bf16(am, pb[j][1], t[j]);
#pragma unroll
        for (int j = 0; j < NB; j++) t[j] = mfma_bf16(ah, pb[j][1], t[j]);
#pragma unroll
        for (int j = 0; j < NB; j++) t[j] = mfma_bf16(am, pb[j][0], t[j]);
#pragma unroll
        for (int j = 0; j < NB; j++) t[j] = mfma_bf16(ah, pb[j][0], t[j]);
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] += t[j];
      }
    }
    __syncthreads();  // the operands have been read
  }

  // acc[i][j][r] = dW[k][channel of a-row (wr*NA + i)*16 + 4*g + r][channel of b-row (wc*NB + j)*16 + r16]
  auto channel = [](int L, int quads) { return 4 * (L % quads) + L / quads; };
  float probe = 0.f;  // stays zero while every sum is finite
#pragma unroll
  for (int i = 0; i < NA; i++)
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) probe = __builtin_fmaf(acc[i][j][r], 0.f, probe);
  if (__ballot(probe != 0.f) != 0ull) {
    // Values that are no finite numbers, or too large for pieces, make the pieces' sums infinite or NaN: the
    // wavefront goes through the share again on the fp32 matrix instructions, 16 positions and one channel per lane and load.
#pragma unroll
    for (int i = 0; i < NA; i++)
#pragma unroll
      for (int j = 0; j < NB; j++) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
    found = 0ull;
    request(0);
    for (int gi = next_granule(); gi < n_granules; gi = next_granule()) {
#pragma unroll
      for (int x = 0; x < 4; x++) {
        const int t = gi * 16 + 4 * g + x;
        int ja = -1, jb = -1;
        if (t < n32) {
          ja = nbr[(int64_t)k * npad + t];
          if (ja >= 0) jb = rowmap ? rowmap[t] : t;
        }
        float va[NA], vb[NB];
#pragma unroll
        for (int i = 0; i < NA; i++) {
          const int c = ca0 + channel((wr * NA + i) * 16 + r16, 8 * NA);
          va[i] = ja >= 0 && c < n_a ? a[(int64_t)ja * n_a + c] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < NB; j++) {
          const int c = cb0 + channel((wc * NB + j) * 16 + r16, 8 * NB);
          vb[j] = jb >= 0 && c < n_b ? b[(int64_t)jb * n_b + c] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < NA; i++)
#pragma unroll
          for (int j = 0; j < NB; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[i], vb[j], acc[i][j], 0, 0, 0);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < NA; i++)
#pragma unroll
      for (int j = 0; j < NB; j++) acc[i][j] *= SPLIT_UNSCALE;
  }
  float *pk = partial + ((size_t)share * K + k) * (size_t)n_a * n_b;
#pragma unroll
  for (int i = 0; i < NA; i++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int c = ca0 + channel((wr * NA + i) * 16 + 4 * g + r, 8 * NA);
      if (c >= n_a) continue;
#pragma unroll
      for (int j = 0; j < NB; j++) {
        const int o = cb0 + channel((wc * NB + j) * 16 + r16, 8 * NB);
        if (o < n_b) pk[(size_t)c * n_b + o] = acc[i][j][r];
      }
    }
}

// Shares of the weight gradient's partial sums written to `partial` ([shares][K][n_a][n_b]), or 0 where the
// kernel does not serve the shape.
int64_t conv_dw_split(Metadata &m, const Table &t, const float *a, int64_t a_rows, int n_a, const float *b, int64_t b_rows,
                      int n_b, hipStream_t s) {
  if (n_a % 4 || n_b % 4 || (uintptr_t)a % 16 || (uintptr_t)b % 16 || t.npad % 4) return 0;
  if (a_rows * n_a * 4 >= ((int64_t)1 << 31) || b_rows * n_b * 4 >= ((int64_t)1 << 31) ||
      (int64_t)t.K * t.npad * 4 >= ((int64_t)1 << 31))
    return 0;
  // Where the other kernels are faster (us, kernel and sums, room surfaces):
  //   a side of up to 32 channels (a million sites 64 x 32 671 there, 722 here; 32 x 32 471 / 651, both in the
  //     narrowest tile that is built, 64 x 64), small levels of up to 64 (20 k 48 x 48 35 / 39)
  //   more than 32 taps: no granule masks, so that a workgroup here stages every granule for every tap (5^3, 5 k sites
  //     64 x 96 159 / 178, 192 x 192 770 / 987, but 128 x 128 378 / 333; 7^3, 20 k 128 x 128 2770 / 5107)
  //   large transposed tables of many taps: few of a position's rows are read twice (400 k fine sites, filter 3 stride 2, 64 x 96
  //     351 / 463, 128 x 128 745 / 796)
  // Up to 32 taps the others wait for a new table's rule counts, which drains the queue: sides of 36 and 48 channels stay here although
  // the tile of 48 is faster by itself (60 k 36 x 36 76 / 92, 48 x 96 132 / 163; but the training step of a U-Net with 24 planes on
  // 150 k sites, new scene each, 7.26 ms with it and 7.09 without, 400 k 11.20 / 11.14), and so do large filter = stride tables
  // (400 k 64 x 64 152 / 165, 96 x 64 144 / 149, 128 x 128 386 / 347).
  const bool transposed = a_rows < t.n;
  if (n_a <= 32 || n_b <= 32 || (t.n < 30000 && n_a <= 64 && n_b <= 64)) return 0;
  if (t.K > 32 || (transposed && t.n >= 300000 && t.K > 9)) return 0;
  // 32 N channels per side: the fewest channels staged, a tile counted as 32 wider than it is
  auto width = [](int planes) {
    int best = 2;
    for (int w = 3; w <= 4; w++)
      if (ceil_div(planes, 32 * w) * (w + 1) <= ceil_div(planes, 32 * best) * (best + 1)) best = w;
    return best;
  };
  const int na = width(n_a), nb = width(n_b);
  const int64_t mt = ceil_div(n_a, 32 * na) * ceil_div(n_b, 32 * nb), per_share = (int64_t)t.K * n_a * n_b;
  // Many shares even out the taps (the centre has 4-7 times the rules of a corner), few leave less to
  // add up: kernel + sums at 1024 / 2048 / 4096 / 8192 / 16384 workgroups, a million sites 64 x 64 1354 / 1149 / 959 /
  // 903 / 945 us, 247 k 362 / 294 / 261 / 278 / 341, 61 k 192 x 96 376 / 300 / 304 / 331 / 465; 14 k 128 x 128 87 at 64 MB
  // of partial sums, 108 at 128.
  // Where a position has few rules, the sums weigh more than evenness does: one tap (1x1 convolutions), 512 / 1024 / 2048 /
  // 8192 workgroups, 400 k rows 64 x 96 108 / 118 / 136 / 162 us, 128 x 128 153 / 173 / 204 / 249; transposed tables
  // and up to nine taps 1024 / 2048 / 4096 / 8192, 60 k sites 96 x 64 61 / 60 / 75 / 76, 2^3 / stride 2 400 k 99 / 99 / 120 / 146,
  // large 2-D levels 400 k 64 x 96 463 / 404 / 386 / 433.
  const bool large = t.n >= 300000, small = t.n < 30000, few_rules = t.K <= 9 || transposed;
  const int workgroups = t.K == 1 ? 512 : few_rules ? (large && !transposed ? 4096 : 2048) : large ? 8192 : small ? 2048 : 4096;
  int64_t shares = ceil_div(workgroups, t.K * mt);
  shares = std::min(shares, std::max<int64_t>(1, ((int64_t)(large ? 256 : small ? 64 : 128) << 18) / per_share));
  shares = std::max<int64_t>(1, std::min(shares, ceil_div(t.n, 16 * DS_BLOCK)));
  const int64_t groups = round_up(shares, 8) * t.K * mt;
  if (groups >= ((int64_t)1 << 31)) return 0;
  m.partial.reserve((size_t)(shares * per_share));
  const unsigned *gm = (t.K <= 32 && t.gmask.p) ? t.gmask.p : nullptr;
  auto launch = [&](auto na_c, auto nb_c) {
    k_conv_dw_split<decltype(na_c)::value, decltype(nb_c)::value><<<dim3((unsigned)groups), 256, 0, s>>>(
        t.nbr.p, t.rowmap_ptr(), gm, t.K, t.n, t.npad, a, n_a, (unsigned)(a_rows * n_a * 4), b, n_b,
        (unsigned)(b_rows * n_b * 4), (int)shares, t.spread ? 1 : 0, m.partial.p);
  };
  auto by_b = [&](auto na_c) {
    if (nb == 2) launch(na_c, std::integral_constant<int, 2>());
    else if (nb == 3) launch(na_c, std::integral_constant<int, 3>());
    else launch(na_c, std::integral_constant<int, 4>());
  };
  if (na == 2) by_b(std::integral_constant<int, 2>());
  else if (na == 3) by_b(std::integral_constant<int, 3>());
  else by_b(std::integral_constant<int, 4>());
  LAUNCH_CHECK();
  return shares;
}

}  // namespace scn
