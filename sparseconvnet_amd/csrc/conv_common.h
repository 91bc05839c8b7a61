// Shared by the translation units of the convolution forward (conv.hip: scratch, weight packing,
// dispatch; conv_tiled.hip, conv_rows.hip, conv_resident.hip: one MFMA kernel family each).
#pragma once
#include "metadata.h"

#include <type_traits>

namespace scn {

// Scratch of a convolution (see conv.hip): buffers of the handle, or fixed regions of the static
// array while an allocation-free call runs.
constexpr size_t NOALLOC_QUEUE_BYTES = 4096;              // set counters (8 x 128 bytes used)
constexpr size_t NOALLOC_WPACK_BYTES = (size_t)8 << 20;   // packed weights: 27 taps of 256 x 256 are 7.1 MB
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)16 << 20;
constexpr size_t NOALLOC_PARTIAL_BYTES = NOALLOC_SCRATCH_BYTES - NOALLOC_WPACK_BYTES - NOALLOC_QUEUE_BYTES;
float *scratch_wpack(Metadata &m, size_t floats);
int *scratch_queue(Metadata &m, hipStream_t s);
float *scratch_partial(Metadata &m, int &n_split, int64_t split_stride_floats);

// The weights of the running convolution in the layout `key` names, `floats` long: from the
// caller's frozen set when there is one (packed by `pack(dst)` the first time), else packed into
// the handle's scratch on every call.
template <class F>
static float *packed_weights(Metadata &m, std::vector<int64_t> key, size_t floats, F pack) {
  auto first = [&] {
    if (m.before_pack) m.before_pack();
    m.before_pack = nullptr;
  };
  if (m.frozen && !m.fixed_scratch) {
    if (m.wkey_ptr) {  // a column range: keyed by where it lies in the caller's weights, not by the scratch copy's address
      key[1] += m.wkey_ptr - m.wkey_from;
      key.push_back(m.wkey_c0);
      key.push_back(m.wkey_wc);
    }
    auto it = m.frozen->packed.find(key);
    if (it != m.frozen->packed.end() && it->second.cap >= floats) return it->second.p;
    DevBuf<float> &b = m.frozen->packed[key];
    b.reserve(floats);
    first();
    pack(b.p);
    return b.p;
  }
  float *dst = scratch_wpack(m, floats);
  first();
  pack(dst);
  return dst;
}

typedef float v4f __attribute__((ext_vector_type(4)));
// Four bf16 values in two registers: the A / B operand of v_mfma_f32_16x16x16_bf16, which
// contracts the 16 channels that four fp32 MFMAs (16x16x4) take one after the other.  A lane
// holds the same four consecutive channels in both layouts, so the reduced-precision kernels
// differ from the fp32 ones only in a conversion (round to nearest even) where operands enter
// LDS or the A registers, and in one MFMA instead of four.
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
__device__ inline v4s to_bf16x4(v4f v) { return __builtin_bit_cast(v4s, __builtin_convertvector(v, v4bf)); }
// The bf16 kernels take two 16-channel steps per v_mfma_f32_16x16x32_bf16: lane group g
// contributes its four channels of either step (the instruction sums over all 32 (lane group,
// element) pairs, in whatever order A and B agree on).  Operands of a pair of steps are kept
// next to each other (16 bytes per lane) in LDS and in the packed weights, so that they
// arrive in the four consecutive registers the instruction wants.
__device__ inline v8s to_bf16x8(v4f lo, v4f hi) {
  return __builtin_shufflevector(to_bf16x4(lo), to_bf16x4(hi), 0, 1, 2, 3, 4, 5, 6, 7);
}
__device__ inline v4f mfma_bf16(v8s a, v8s b, v4f acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), acc, 0, 0, 0);
}

// ---- fp32 operands as three bf16 pieces -------------------------------------------------
// x = h + m + l, each rounded to the eight bits of bf16 (G. Henry, P. T. P. Tang, A. Heinecke, "Leveraging the
// bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", ARITH 2019).  For x in [2^e, 2^(e+1))
// |m| <= 2^(e-8) and |l| <= 2^(e-17), so that of the nine products of two such numbers h l' + l h' + m m' and above
// count and m l' + l m' + l l' <= 1.001 2^-24 2^(e+e') are left out (cut off instead of rounded, h would leave
// an m of up to 2^(e-7) and four times as much: single products up to 4.8 2^-24 off, against 2.4 now and 1.0 on the
// fp32 matrix instructions, which round to nearest).  The other six are one
// v_mfma_f32_16x16x32_bf16 each, 96 cycles of the matrix unit for 32 channels where eight
// v_mfma_f32_16x16x4_f32 take 256.  (The matrix unit sustains 1700 TFLOP/s on the former and 140
// on the latter, operands in registers: twice the rate after the six-fold work.)
// The six products of 32 channels are summed from zero and then added to the accumulator in fp32: a
// chain of them straight into the accumulator rounds with the accumulator's exponent every time, and
// not to nearest.  Against sums in 64 bits, 16 x 16 tiles, 1728 channels (relative 2-norm): fp32
// matrix instructions 7.5e-7 (signed values) / 5.3e-7 (ReLU outputs) / 4.2e-7 (all positive), six
// products into the accumulator 6.4e-7 / 6.2e-7 / 7.7e-7, summed apart 1.5e-7 / 1.5e-7 / 1.1e-7.
// The pieces are those of 2^24 x: bf16 ends at 2^-133 where fp32 ends at 2^-149, and pieces of x itself would lose bits of
// every x below 2^-110 (4.7e-2 of the result at 2^-126, all of it at 2^-140).  Sums of products come out 2^48 times too
// large (SPLIT_UNSCALE).  (Costs a multiplication per value staged: a stack of layers at a million sites 10.13 -> 10.19 ms,
// training step 24.8 -> 24.9, narrow layers 2 % (32 -> 32 at a million sites 254 -> 260 us, 250 k 128 -> 32 239 -> 245).
// v_dot2_f32_bf16 in place of unpacking and subtracting the pieces is neither exact nor faster.)
// A number that no bf16 then rounds (2e31 and more) has infinite pieces: whoever multiplies them, or has a sum past
// 1.2e24, finds a sum that is not finite and computes it in fp32.
constexpr float SPLIT_SCALE = 0x1p24f, SPLIT_UNSCALE = 0x1p-48f;
__device__ inline void split_pair(float x0, float x1, unsigned &h, unsigned &m, unsigned &l) {
  typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
  typedef float v2f __attribute__((ext_vector_type(2)));
  x0 *= SPLIT_SCALE, x1 *= SPLIT_SCALE;
  h = __builtin_bit_cast(unsigned, __builtin_convertvector((v2f){x0, x1}, v2bf));
  const float r0 = x0 - __builtin_bit_cast(float, h << 16), r1 = x1 - __builtin_bit_cast(float, h & 0xFFFF0000u);
  m = __builtin_bit_cast(unsigned, __builtin_convertvector((v2f){r0, r1}, v2bf));
  const float l0 = r0 - __builtin_bit_cast(float, m << 16), l1 = r1 - __builtin_bit_cast(float, m & 0xFFFF0000u);
  l = __builtin_bit_cast(unsigned, __builtin_convertvector((v2f){l0, l1}, v2bf));
}
// Packed weights: the pieces of v, or, of a number that has none, an infinity and its own two halves.
constexpr short PIECE_WHOLE = 0x7F80;
__device__ inline void split_weight(float v, short &h, short &m, short &l) {
  unsigned ph, pm, pl;
  split_pair(v, 0.0f, ph, pm, pl);
  const bool whole = (ph & 0x7F80u) == 0x7F80u;
  const unsigned u = __builtin_bit_cast(unsigned, v);
  h = whole ? PIECE_WHOLE : (short)ph;
  m = (short)(whole ? u >> 16 : pm);
  l = (short)(whole ? u : pl);
}
__device__ inline float join_weight(short h, short m, short l) {
  auto upper = [](short b) { return (unsigned)(unsigned short)b << 16; };
  if (h == PIECE_WHOLE) return __builtin_bit_cast(float, upper(m) | (unsigned short)l);
  return ((__builtin_bit_cast(float, upper(h)) + __builtin_bit_cast(float, upper(m))) + __builtin_bit_cast(float, upper(l))) *
         (1.0f / SPLIT_SCALE);
}
struct Split8 {  // eight channels of a lane: the operands of the three pieces
  v8s h, m, l;
};
__device__ inline Split8 split8(v4f a, v4f b) {
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  unsigned h[4], m[4], l[4];
  split_pair(a.x, a.y, h[0], m[0], l[0]);
  split_pair(a.z, a.w, h[1], m[1], l[1]);
  split_pair(b.x, b.y, h[2], m[2], l[2]);
  split_pair(b.z, b.w, h[3], m[3], l[3]);
  Split8 s;
  s.h = __builtin_bit_cast(v8s, (v4u){h[0], h[1], h[2], h[3]});
  s.m = __builtin_bit_cast(v8s, (v4u){m[0], m[1], m[2], m[3]});
  s.l = __builtin_bit_cast(v8s, (v4u){l[0], l[1], l[2], l[3]});
  return s;
}

template <bool PRE> __device__ inline v4f pre_act(v4f v, v4f sc, v4f sh, float leak) {
  if (!PRE) return v;
  v4f y = v * sc + sh;
  y.x *= (y.x > 0.f ? 1.f : leak);
  y.y *= (y.y > 0.f ? 1.f : leak);
  y.z *= (y.z > 0.f ? 1.f : leak);
  y.w *= (y.w > 0.f ? 1.f : leak);
  return y;
}
// Hands the pending jobs to the launch being prepared (and forgets them).
static inline CoefJobs take_jobs(Metadata &m) {
  CoefJobs j = m.jobs;
  m.jobs = CoefJobs();
  return j;
}

// Elements of one packed weight slab (SS steps of 16 channels by NCB column blocks), padded to
// a multiple of 256 lanes' worth so that a workgroup stages it without bounds checks.
constexpr int packed_slab_floats(int SS, int NCB) { return (SS * NCB * 64 + 255) / 256 * 256 * 4; }


// Profiling build (-DSCN_PHASES, see build.py's SCN_EXTRA_FLAGS): thread 0 of every 16th workgroup
// of a tiled kernel stamps the 100 MHz wall clock at up to seven points of its life into its
// translation unit's g_phase_stamps; slot 7 holds the tile's iteration count.  SCN_PHASE_EXPORT(name)
// defines the extern "C" function that copies the stamps to the host.  Compiled out otherwise.
#ifdef SCN_PHASES
static __device__ unsigned long long g_phase_stamps[64 * 8];
#define SCN_PHASE_SLOT() (blockIdx.y == 0 && (blockIdx.x % 16) == 0 && blockIdx.x / 16 < 64 && threadIdx.x == 0)
#define SCN_PHASE(i) do { if (SCN_PHASE_SLOT()) g_phase_stamps[(blockIdx.x / 16) * 8 + (i)] = wall_clock64(); } while (0)
#define SCN_PHASE_VALUE(i, v) do { if (SCN_PHASE_SLOT()) g_phase_stamps[(blockIdx.x / 16) * 8 + (i)] = (unsigned long long)(v); } while (0)
#define SCN_PHASE_EXPORT(name) \
  extern "C" int name(unsigned long long *out) { return (int)hipMemcpyFromSymbol(out, HIP_SYMBOL(g_phase_stamps), sizeof(g_phase_stamps)); }
#else
#define SCN_PHASE(i)
#define SCN_PHASE_VALUE(i, v)
#define SCN_PHASE_EXPORT(name)
#endif

// Notes the kernel a convolution call launches (Metadata::last_kernel).
inline void note_kernel(Metadata &m, const char *family, std::initializer_list<std::pair<const char *, int>> params) {
  std::string t = family;
  for (auto &p : params) t += std::string(" ") + p.first + "=" + std::to_string(p.second);
  if (!m.last_kernel.empty() && m.last_kernel.back() == '+') m.last_kernel += " " + t;  // column ranges, channel parts
  else m.last_kernel = t;
}

struct PreArgs {  // device pointers to the padded coefficient arrays, or nulls
  const float *sc = nullptr, *sh = nullptr;
  float leak = 1.0f;
};

// What a tile's workgroup (NT threads, G granules of 16 positions from position tbase on) sets up
// before its tap loop: the tile's neighbour rows in LDS, jtab[(granule * K + tap) * 16 + row], the
// granules that have each tap, gmask[tap], and the list of the taps any of its rows has (of those
// this workgroup is to take when the taps of a tile are dealt over n_split workgroups: tap k
// belongs to workgroup k % n_split, or, RANKED, a tile's i-th tap to workgroup i % n_split, which keeps the parts even
// where a tile's taps are those of one parity: fine side of filter 3 stride 2, 8 k sites 64 -> 64 22.4 -> 19.7 us,
// 128 -> 96 26.1).  Every thread of the workgroup calls it; it ends with a
// barrier and returns the length of the list.
// The table is read tap by tap, 16 * G consecutive entries each, and all of a thread's loads
// (up to eight) are in flight together: a loop of load - store - ballot steps paid one memory
// latency per step, 5 us for 27 taps where the whole convolution of a small level takes 20.
template <int NT, int G, bool RANKED = false>
__device__ inline int tile_setup(const int *__restrict__ nbr, int K, int64_t n, int64_t npad, int64_t tbase, int n_split,
                                 int split, int *jtab, unsigned *gmask, int *taplist, int *ntaps_p) {
  constexpr int PER_TAP = G * 16;          // entries of one tap
  static_assert(NT % PER_TAP == 0 || PER_TAP % NT == 0, "threads and tile rows must divide one another");
  for (int k = threadIdx.x; k < K; k += NT) gmask[k] = 0u;
  __syncthreads();
  const int total = K * PER_TAP;
  constexpr int BATCH = 8;
  for (int e0 = 0; e0 < total; e0 += BATCH * NT) {
    int jv[BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; i++) {
      const int e = e0 + i * NT + (int)threadIdx.x;
      const int k = e / PER_TAP, p = e % PER_TAP;
      jv[i] = -1;
      if (e < total && tbase + p < n) jv[i] = nbr[(int64_t)k * npad + tbase + p];
    }
#pragma unroll
    for (int i = 0; i < BATCH; i++) {
      const int e = e0 + i * NT + (int)threadIdx.x;
      const int k = e / PER_TAP, p = e % PER_TAP;
      if (e < total) jtab[((p >> 4) * K + k) * 16 + (p & 15)] = jv[i];
      // sixteen consecutive lanes hold one granule's rows of one tap
      const unsigned long long bal = __ballot(jv[i] >= 0);
      const int lane = threadIdx.x & 63;
      if ((lane & 15) == 0 && e < total && ((bal >> lane) & 0xFFFFull)) atomicOr(&gmask[k], 1u << (p >> 4));
    }
  }
  __syncthreads();
  if (threadIdx.x < 64) {  // the first wavefront lists the taps, 64 at a time, in ascending order
    int count = 0;
    for (int k0 = 0; k0 < K; k0 += 64) {
      const int k = k0 + (int)threadIdx.x;
      const bool mine = k < K && gmask[k] != 0u && (RANKED || n_split == 1 || k % n_split == split);
      const unsigned long long bal = __ballot(mine);
      const int rank = count + __popcll(bal & ((1ull << threadIdx.x) - 1ull));
      if (!RANKED && mine) taplist[rank] = k;
      if (RANKED && mine && rank % n_split == split) taplist[rank / n_split] = k;
      count += __popcll(bal);
    }
    if (threadIdx.x == 0) *ntaps_p = RANKED ? (count + n_split - 1 - split) / n_split : count;
  }
  __syncthreads();
  return *ntaps_p;
}

// Launchers of the kernels conv.hip defines for the other translation units.
// k_pack_weights / k_pack_weights_part / k_pack_weights_c4: weights into MFMA B-operand order.
void launch_pack_weights(const float *w, float *wp, int K, int n_in, int n_out, int n_slab, int SS, int NCB,
                         int slab_stride, CoefJobs jobs, bool as_bf16, hipStream_t s);
void launch_pack_weights_part(const float *w, float *wp, int K, int w_rows, int n_in_part, int n_out, int SS, int NCB,
                              int *queue, CoefJobs jobs, bool as_bf16, hipStream_t s);
void launch_pack_weights_c4(const float *w, float *wp, int K, int n_in, int n_out, int NCB, int *queue, CoefJobs jobs,
                            hipStream_t s);
// out[rowmap[pos]][col] = epilogue(bias[col] + sum over splits of partial[split][pos][col])
void launch_conv_reduce(const float *partial, int n_split, int64_t split_stride, int ld, const int *rowmap, int64_t n,
                        Epi epi, float *out, int n_out, hipStream_t s);

// The three MFMA kernel families; each returns false when it has no instantiation for the shape.
bool conv_tiled_dispatch(bool vec4, bool pre_fused, Metadata &m, const Table &t, const float *in, float *out,
                         const float *w, Epi epi, int n_in, int n_out, PreArgs pre, hipStream_t s);
bool conv_rows_dispatch(bool vec4, bool pre_fused, Metadata &m, const Table &t, const float *in, float *out,
                        const float *w, Epi epi, int n_in, int n_out, PreArgs pre, hipStream_t s);
// conv_split.hip: fp32 operands as three bf16 pieces each.
bool conv_split_serves(const Metadata &m, const Table &t, const float *in, int64_t in_rows, int n_in, int n_out);
bool conv_split_dispatch(bool pre_fused, Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi,
                         int n_in, int n_out, PreArgs pre, hipStream_t s);
const float *split_weights(Metadata &m, int K, const float *w, int n_in, int n_out, int NCB, bool half, hipStream_t s);
// conv_wave.hip: the same for up to 48 output planes.  gradient: an input gradient over the table (weights packed transposed).
bool conv_wave_serves(const Metadata &m, const Table &t, const float *in, int64_t in_rows, int n_in, int n_out, bool gradient = false);
bool conv_wave_dispatch(bool pre_fused, Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi,
                        int n_in, int n_out, PreArgs pre, hipStream_t s);
// conv_few.hip: transposed convolutions of filter = stride = 2 rulebooks whose weights fit LDS.
bool try_few(Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi, int n_in, int n_out,
             hipStream_t s);
bool resident_fits(const Metadata &m, const Table &t, int n_in, int n_out, bool with_bn);
bool try_resident(Metadata &m, const Table &t, const float *in, float *out, const float *w, Epi epi, int n_in,
                  int n_out, hipStream_t s);

}  // namespace scn
