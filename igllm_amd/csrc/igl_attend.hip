// igl_attend.hip - decode attention over the byte-quantized key/value ring,
// gfx950.
//
// For one lane (one query position) and each key/value head shared by 8
// query heads, computes
//     o_h = sum_t softmax_t(score_scale * q_h . k_t) v_t
// over the visible positions t = place_start .. place_start + span - 1, whose
// rows sit in ring slot t % cache_span (session_attend_group with
// attend_score_band and attend_blend_band, app_core.c:11296-11453; ring and
// span rules 11500, 11516-11526).  A stored byte decodes to
//     e4m3:  cache_real8(byte) * scale   (cache_real8, app_core.c:11018-11030)
//     int8:  (int8_t)byte * scale
// The reference scores every row against `grid[byte] = real8 * scale`; here
// the scale multiplies the finished dot product, the same value up to fp32
// rounding.
//
// Why MFMA: with 8 query heads on one key/value head every key and value
// byte feeds 8 multiply-adds, 8 MAC per byte of HBM traffic, above the ~5
// fp32 MAC per byte the vector ALU can sustain at the HBM rate.  Both
// products therefore run on v_mfma_f32_16x16x32_f16:
//   scores  S[16 x 32 positions] = [q_hi; q_lo] (16 x d) . K^T (d x 32)
//   blend   O[16 x d]            = [p_hi; p_lo] (16 x 32) . V (32 x d)
// The 16 MFMA rows hold each head twice, as an exact two-term binary16 split
// (x = hi + lo, |lo| <= 2^-11 |x|), so the products keep ~22 significant
// bits and accumulate in fp32; the two rows are added at the end.  Bytes
// decode to binary16 exactly:
//   e4m3: move bit 7 to bit 8 and shift the byte up by 7, giving
//         real8(byte) / 256 for all 256 codes (0x7F/0xFF read +-480, as the
//         reference reads them);
//   int8: (byte ^ 0x80) in the mantissa of 1024.0, minus 1152.
//
// Work layout (flash-decoding): a lane's span is cut into chunks of C
// positions (32 up to kAttendShortSpan, 64 beyond), one workgroup of four
// waves a chunk.  The two products split the chunk differently among the
// waves, so each wave's dependent chain is a quarter of the chunk's work:
// scores by positions (wave w: C/4 positions over every dim), the blend by
// dims (wave w: a quarter of the dims over every position).  A span of one
// chunk is written directly; otherwise each chunk writes a partial (blend,
// peak, total) and attend_fold_kernel folds them in one memory round trip.
//
// (Measured on the box, one launch pair inside a graph: a 512-position
// sliding window of 256-dim heads takes 9.5 us, of which 4.9 us is the chunk
// kernel and 1.55 us the bare cost of each dependent launch; the former form,
// one wave per 32 positions over every dim with a cross-wave merge, took 6.9
// us for the same chunks.  A last-workgroup fold in the same kernel, after an
// agent-scope release/acquire ticket, was slower at every chunk count tried:
// 10.5 us at 8 chunks, over 100 us at 256.)
#include <mutex>

#include "igl_backend.h"
#include "igl_device.h"

namespace igl {

// Positions a chunk, by the longest span a launch covers: 32 up to
// kAttendShortSpan (the most workgroups, the shortest chain each), 64 beyond
// (half the partials: at 16384 positions 11.4 us against 13.0 us for 32).
// One lane's sliding window measured 6.8 us with 32 against 7.3 with 64.
// Launches of kAttendWideLanes lanes and more (a prefill pass) take 64 whatever
// the span: those of one chunk keep no partials, the others take tiles of lanes.
constexpr int kAttendShortSpan = 8192;
constexpr int kAttendWideLanes = 64;
constexpr int kAttendGroup = 8;                    // query heads per key/value head
constexpr int kAttendPrepLanes = 4;                // lanes of one prepared launch

struct AttendArgs {
  const uint8_t *key_store;    // [cache_span][kv_width]
  const uint8_t *value_store;
  int kv_width;
  int cache_span;
  int place0;                  // position of lane 0; lane l is at place0 + l
  const int *place_dev;        // when set, lane 0's position is read here instead
  int window;                  // positions a lane sees (0: all from position 0)
  int chunks;                  // workgroup slots per lane in the partial buffers
  float *final_out;            // when one workgroup covers a lane: the blend, [lanes][q_stride]
  int q_stride;                // floats between lanes of query / blend
  const float *query;          // [lanes][head_count][HEAD]
  float key_scale;             // decoded-byte multiplier, score_scale folded in
  float value_scale;
  float *part_out;             // [chunks][head_count][HEAD]
  float *part_peak;            // [chunks][head_count]; of a tile, log2
  float *part_total;           // [chunks][head_count]
  int head_count;
  // The heads of a decode step or a small block prepared here
  // (attend_split_kernel's PREP form): `query` holds the query heads before
  // their norm; q_gain their gain; turn, lane by lane, the (cos, sin) of the
  // lane's position times each rotation step, HEAD / 2 pairs.  With k_raw
  // set, the block's new positions place .. place + l (lane l's, and the
  // lanes' before it) get a workgroup of lane l's own after the chunks of the
  // positions before the block (attend_fresh_rows): it prepares their key and
  // value heads (norm and gain and turn; norm), writes lane l's bytes into
  // ring slot (place + l) % cache_span of k_ring / v_ring (the rings read
  // here), code = e4m3(value / scale), and writes the partial of those
  // positions; the chunk workgroups never read those slots.
  const float *q_gain;
  const float *turn;           // [lanes][HEAD / 2][2]
  int turn_stride;             // floats between lanes of turn
  const float *k_raw;          // [lanes][kv_raw_stride], as v_raw
  int kv_raw_stride;
  const float *v_raw;
  const float *k_gain;
  uint8_t *k_ring;
  uint8_t *v_ring;
  float k_code_scale;
  float v_code_scale;
  float eps;
  int lanes;                   // of the launch (tiles)
};

// Two bytes held in bits [0,8) and [16,24) of `x`, as two exact binary16.
template <int FMT>
__device__ __forceinline__ uint32_t decode_pair(uint32_t x) {
  if (FMT == 0) {
    return (x + (x & 0x00800080u)) << 7;  // e4m3 -> real8 / 256
  } else {
    half2_t h = as_half2(x ^ 0x64806480u);  // 1152 + (int8)byte
    h = h + half2_t{(_Float16)-1152.0f, (_Float16)-1152.0f};
    return __builtin_bit_cast(uint32_t, h);
  }
}

// Eight bytes (two dwords, low byte first) as eight binary16 operand values.
template <int FMT>
__device__ __forceinline__ half8_t decode8(uint32_t lo, uint32_t hi) {
  uint32_t w[4];
  w[0] = decode_pair<FMT>(__builtin_amdgcn_perm(0u, lo, 0x0C010C00u));
  w[1] = decode_pair<FMT>(__builtin_amdgcn_perm(0u, lo, 0x0C030C02u));
  w[2] = decode_pair<FMT>(__builtin_amdgcn_perm(0u, hi, 0x0C010C00u));
  w[3] = decode_pair<FMT>(__builtin_amdgcn_perm(0u, hi, 0x0C030C02u));
  return __builtin_bit_cast(half8_t, w);
}

// v plus its partner 32 lanes away, the same value in both lanes: one
// v_permlane32_swap of two copies of v leaves the lower halves in one and the
// upper halves in the other.  Written out because the builtin given the same
// value twice is folded as if both results were its first; the s_nops are the
// waits the compiler itself places around this instruction.
__device__ __forceinline__ float xsum32(float v) {
  float lo = v, hi = v;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(lo), "+v"(hi));
  return lo + hi;
}

// The block's new positions seen by lane l, pos0 .. pos0 + l, a workgroup of
// the lane's own (PREP with k_raw): the key and value heads of each new
// position prepared (norm, gain, turn; norm), lane l writing only its own
// position's bytes to the rings (lanes before it write theirs, from the same
// arithmetic on the same inputs); the lane's 8 query heads prepared as every
// chunk prepares them; and one partial over those l + 1 positions: score_h,j
// = key_scale q_h . key_j(bytes) in fp32, peak_h = max_j score_h,j, total_h =
// sum_j e^(score_h,j - peak_h), blend_h = sum_j e^(score_h,j - peak_h)
// value_j(bytes) value_scale (one position: peak = its score, total 1, blend
// its value).  Off the path of the chunk workgroups, which end before it.
template <int HEAD>
__device__ __forceinline__ void attend_fresh_rows(const AttendArgs &a, int pos0, int l, int pc) {
  constexpr int HALF = HEAD / 2;
  constexpr int W = 4;
  constexpr int F = kAttendPrepLanes;
  constexpr int kHeadItems = HEAD / 8;
  constexpr int kQItems = kAttendGroup * HEAD / 8 / 256;
  __shared__ double nr_red[F][2][W];
  __shared__ __attribute__((aligned(16))) uint8_t nr_bytes[F][2][HEAD];
  __shared__ float nr_score[kAttendGroup][F];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int rows = l + 1;  // uniform, at most F
  // every load first: the key/value pairs of the thread (threads below
  // HALF) of each new position, then its query items with their gains and
  // turns
  float kx[F][2], vx[F][2], kt[F][2], kg[2] = {0.0f, 0.0f};
#pragma unroll
  for (int j = 0; j < F; ++j) {
    kx[j][0] = kx[j][1] = vx[j][0] = vx[j][1] = kt[j][0] = kt[j][1] = 0.0f;
  }
  if (tid < HALF) {
    kg[0] = a.k_gain[tid];
    kg[1] = a.k_gain[tid + HALF];
#pragma unroll
    for (int j = 0; j < F; ++j) {
      if (j < rows) {
        const float *kr = a.k_raw + (size_t)j * a.kv_raw_stride;
        const float *vr = a.v_raw + (size_t)j * a.kv_raw_stride;
        const float *tr = a.turn + (size_t)j * a.turn_stride;
        kx[j][0] = kr[tid];
        kx[j][1] = kr[tid + HALF];
        vx[j][0] = vr[tid];
        vx[j][1] = vr[tid + HALF];
        kt[j][0] = tr[2 * tid];
        kt[j][1] = tr[2 * tid + 1];
      }
    }
  }
  float qf[kQItems][8];
  float4_t qgain[kQItems][2], qturn[kQItems][4];
  const float *own_turn = a.turn + (size_t)l * a.turn_stride;
#pragma unroll
  for (int i = 0; i < kQItems; ++i) {
    const int item = tid + 256 * i;
    const float4_t *q = reinterpret_cast<const float4_t *>(a.query + (size_t)l * a.q_stride + 8 * item);
    const float4_t u = q[0], v = q[1];
    qf[i][0] = u.x; qf[i][1] = u.y; qf[i][2] = u.z; qf[i][3] = u.w;
    qf[i][4] = v.x; qf[i][5] = v.y; qf[i][6] = v.z; qf[i][7] = v.w;
    const int d0 = 8 * (item % kHeadItems);
    const int j0 = d0 < HALF ? d0 : d0 - HALF;
    qgain[i][0] = *reinterpret_cast<const float4_t *>(a.q_gain + d0);
    qgain[i][1] = *reinterpret_cast<const float4_t *>(a.q_gain + d0 + 4);
#pragma unroll
    for (int w = 0; w < 4; ++w) qturn[i][w] = *reinterpret_cast<const float4_t *>(own_turn + 2 * j0 + 4 * w);
  }
  // keys: norm, gain, turn; values: norm (session_attend 11504-11510), every
  // new position's sums behind one barrier
  {
#pragma unroll
    for (int j = 0; j < F; ++j) {
      if (j < rows) {
        double ks = (double)kx[j][0] * (double)kx[j][0] + (double)kx[j][1] * (double)kx[j][1];
        double vs2 = (double)vx[j][0] * (double)vx[j][0] + (double)vx[j][1] * (double)vx[j][1];
        ks = wave_sum_f64_to_last(ks);
        vs2 = wave_sum_f64_to_last(vs2);
        if (lane == 63) {
          nr_red[j][0][wave] = ks;
          nr_red[j][1][wave] = vs2;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < F; ++j) {
      if (j < rows) {
        double kt_sum = nr_red[j][0][0], vt_sum = nr_red[j][1][0];
#pragma unroll
        for (int w = 1; w < W; ++w) {
          kt_sum += nr_red[j][0][w];
          vt_sum += nr_red[j][1][w];
        }
        if (tid < HALF) {
          const float ksh = rms_shrink(kt_sum, HEAD, a.eps);
          const float vsh = rms_shrink(vt_sum, HEAD, a.eps);
          float lo = kx[j][0] * ksh, hi = kx[j][1] * ksh;
          lo = lo * kg[0];
          hi = hi * kg[1];
          const float k0 = lo * kt[j][0] - hi * kt[j][1];
          const float k1 = hi * kt[j][0] + lo * kt[j][1];
          const uint8_t b0 = e4m3_code(k0 / a.k_code_scale), b1 = e4m3_code(k1 / a.k_code_scale);
          const uint8_t c0b = e4m3_code(vx[j][0] * vsh / a.v_code_scale);
          const uint8_t c1b = e4m3_code(vx[j][1] * vsh / a.v_code_scale);
          if (j == l) {
            const size_t row = (size_t)((pos0 + l) % a.cache_span) * a.kv_width;
            a.k_ring[row + tid] = b0;
            a.k_ring[row + tid + HALF] = b1;
            a.v_ring[row + tid] = c0b;
            a.v_ring[row + tid + HALF] = c1b;
          }
          nr_bytes[j][0][tid] = b0;
          nr_bytes[j][0][tid + HALF] = b1;
          nr_bytes[j][1][tid] = c0b;
          nr_bytes[j][1][tid + HALF] = c1b;
        }
      }
    }
  }
  __syncthreads();
  // the query heads as the chunks prepare them, then each item's share of
  // its head's score against each new position's decoded key bytes
#pragma unroll
  for (int i = 0; i < kQItems; ++i) {
    const int item = tid + 256 * i;
    const int h = item / kHeadItems;
    const int d0 = 8 * (item % kHeadItems);
    double ss = 0.0;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += (double)qf[i][e] * (double)qf[i][e];
#pragma unroll
    for (int off = kHeadItems / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
    const float shrink = rms_shrink(ss, HEAD, a.eps);
    const float gg[8] = {qgain[i][0].x, qgain[i][0].y, qgain[i][0].z, qgain[i][0].w,
                         qgain[i][1].x, qgain[i][1].y, qgain[i][1].z, qgain[i][1].w};
    float own[8], other[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      own[e] = qf[i][e] * shrink;
      own[e] = own[e] * gg[e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) other[e] = __shfl_xor(own[e], kHeadItems / 2);
    const bool low = d0 < HALF;
    float qv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float c = qturn[i][e >> 1][2 * (e & 1)];
      const float sn = qturn[i][e >> 1][2 * (e & 1) + 1];
      qv[e] = low ? own[e] * c - other[e] * sn : own[e] * c + other[e] * sn;
    }
#pragma unroll
    for (int j = 0; j < F; ++j) {
      if (j < rows) {
        const uint2_t kb = *reinterpret_cast<const uint2_t *>(&nr_bytes[j][0][d0]);
        const half8_t kd = decode8<0>(kb.x, kb.y);
        float part = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) part = __builtin_fmaf(qv[e], (float)kd[e], part);
#pragma unroll
        for (int off = kHeadItems / 2; off > 0; off >>= 1) part += __shfl_xor(part, off);
        if (item % kHeadItems == 0) nr_score[h][j] = part * a.key_scale;
      }
    }
  }
  __syncthreads();
  // the partial: each head blends the new value rows, weighted against its peak
  for (int i = tid; i < kAttendGroup * HEAD / 8; i += 256) {
    const int h = i / (HEAD / 8);
    const int d0 = 8 * (i % (HEAD / 8));
    float peak = nr_score[h][0];
    for (int j = 1; j < rows; ++j) peak = fmaxf(peak, nr_score[h][j]);
    float o[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    for (int j = 0; j < rows; ++j) {
      const float wgt = __expf(nr_score[h][j] - peak);
      const uint2_t vb = *reinterpret_cast<const uint2_t *>(&nr_bytes[j][1][d0]);
      const half8_t vd = decode8<0>(vb.x, vb.y);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] += wgt * ((float)vd[e] * a.value_scale);
    }
    float *dst = a.part_out + ((size_t)pc * a.head_count + h) * HEAD + d0;
    *reinterpret_cast<float4_t *>(dst) = float4_t{o[0], o[1], o[2], o[3]};
    *reinterpret_cast<float4_t *>(dst + 4) = float4_t{o[4], o[5], o[6], o[7]};
  }
  if (tid < kAttendGroup) {
    float peak = nr_score[tid][0];
    for (int j = 1; j < rows; ++j) peak = fmaxf(peak, nr_score[tid][j]);
    float total = 0.0f;
    for (int j = 0; j < rows; ++j) total += __expf(nr_score[tid][j] - peak);
    a.part_peak[(size_t)pc * a.head_count + tid] = peak;
    a.part_total[(size_t)pc * a.head_count + tid] = total;
  }
}

// The split form.  A workgroup of four waves takes a chunk of C positions
// (32 or 64) of one lane.  The two products are split differently among the
// waves, so that each wave's dependent chain is a quarter of the chunk's work:
//   scores: wave w takes positions w*C/4 .. (w+1)*C/4 - 1 over every dim (its
//           key rows straight into MFMA operand order, as above);
//   blend:  wave w takes dims w*HEAD/4 .. (w+1)*HEAD/4 - 1 over every position
//           of the chunk (its slice of each value row staged in its own LDS).
// Between the two, the probabilities (against each wave's own peak) and the
// waves' peaks and sums go through LDS: one barrier.  Each wave then owns its
// dims of the output outright, so nothing is merged across waves.
template <int HEAD, int FMT, int C, bool QVEC, bool PREP>
__global__ __launch_bounds__(256) void attend_split_kernel(AttendArgs a) {
  constexpr int W = 4;                // waves
  constexpr int PW = C / W;           // positions a wave scores: 8 or 16
  constexpr int DS = HEAD / W;        // dims a wave blends: 64 or 128
  constexpr int S = HEAD / 32;        // k-steps of the score product
  constexpr int QD = HEAD / 4;        // bytes of a key row one lane group reads
  constexpr int QUADS = DS / 64;      // 64-dim groups of a wave's blend
  constexpr int KS = C / 32;          // k-steps of the blend (32 positions each)
  constexpr int VP = DS + 8;          // staged value row pitch in bytes (8-byte aligned rows)
  constexpr int LPR = DS / 16;        // lanes that load one value row (16 bytes each)
  constexpr int RPI = 64 / LPR;       // value rows one load instruction covers
  constexpr int VL = C / RPI;         // value loads a lane issues
  static_assert(PW == 8 || PW == 16, "chunk of 32 or 64 positions");
  static_assert(!PREP || (FMT == 0 && QVEC), "prepared heads: e4m3 rings, aligned queries");
  constexpr int HALF = HEAD / 2;

  __shared__ half8_t qs[2][kAttendGroup][HEAD / 8];
  __shared__ float ps[kAttendGroup][C];
  __shared__ __attribute__((aligned(16))) float wm[W][kAttendGroup];
  __shared__ __attribute__((aligned(16))) float wl[W][kAttendGroup];
  __shared__ __attribute__((aligned(16))) uint8_t vs[W][C * VP];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int g = lane >> 4;
  const int n = lane & 15;
  const int kv = blockIdx.y;
  const int head0 = kv * kAttendGroup;
  const int block = blockIdx.x;
  const int lane_id = blockIdx.z;
  const int pos0 = a.place_dev ? *a.place_dev : a.place0;
  const int pos = pos0 + lane_id;
  const int span_full = a.window > 0 ? min(pos + 1, a.window) : pos + 1;
  const int place_start = pos - span_full + 1;
  // PREP with k_raw: the block's new positions up to the lane's own are the
  // workgroup after the chunks, which cover the positions before the block
  // (lane_id + 1 <= kAttendPrepLanes is inside every window)
  const bool new_row = PREP && a.k_raw != nullptr;
  const int span_count = new_row ? span_full - (lane_id + 1) : span_full;
  const int blocks_seen = (span_count + C - 1) / C;
  const int pc = lane_id * a.chunks + block;
  if (new_row && block == blocks_seen) {
    if (PREP) attend_fresh_rows<HEAD>(a, pos0, lane_id, pc);
    return;
  }
  if (block >= blocks_seen) return;  // past this lane's span: the whole workgroup
  const size_t kv_off = (size_t)kv * HEAD;
  const int c0 = block * C;  // the chunk's first position (relative to place_start)
  // ring slot of relative position t: (place_start + t) % cache_span, from one
  // uniform remainder (0 <= t < span <= cache_span, so one wrap at most)
  const int ring0 = place_start % a.cache_span;
  auto ring_slot = [&](int t) {
    const int slot = ring0 + t;
    return slot >= a.cache_span ? slot - a.cache_span : slot;
  };

  // ---- loads, all issued before the first wait
  constexpr int kQTotal = kAttendGroup * HEAD / 8;
  constexpr int kQItems = kQTotal / 256;
  float qf[kQItems][8];
  {
    const float *qb = a.query + (size_t)lane_id * a.q_stride + (size_t)head0 * HEAD;
#pragma unroll
    for (int i = 0; i < kQItems; ++i) {
      const float *q = qb + 8 * (tid + 256 * i);
      if (QVEC) {
        const float4_t u = *reinterpret_cast<const float4_t *>(q);
        const float4_t v = *reinterpret_cast<const float4_t *>(q + 4);
        qf[i][0] = u.x; qf[i][1] = u.y; qf[i][2] = u.z; qf[i][3] = u.w;
        qf[i][4] = v.x; qf[i][5] = v.y; qf[i][6] = v.z; qf[i][7] = v.w;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[i][e] = q[e];
      }
    }
  }
  // PREP: the gains and turns of the thread's query dims, requested with the
  // query itself (one round trip, not two): item i covers dims d0 .. d0 + 7 of
  // its head, whose turn pairs j0 .. j0 + 7 are 16 consecutive floats.
  constexpr int kHeadItems = HEAD / 8;
  float4_t qgain[PREP ? kQItems : 1][2];
  float4_t qturn[PREP ? kQItems : 1][4];
  if (PREP) {
#pragma unroll
    for (int i = 0; i < kQItems; ++i) {
      const int d0 = 8 * ((tid + 256 * i) % kHeadItems);
      const int j0 = d0 < HALF ? d0 : d0 - HALF;
      qgain[i][0] = *reinterpret_cast<const float4_t *>(a.q_gain + d0);
      qgain[i][1] = *reinterpret_cast<const float4_t *>(a.q_gain + d0 + 4);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        qturn[i][v] = *reinterpret_cast<const float4_t *>(a.turn + (size_t)lane_id * a.turn_stride + 2 * j0 + 4 * v);
    }
  }
  // key row: position c0 + wave*PW + (n % PW), bytes QD*g .. QD*g + QD - 1
  const int tk = c0 + wave * PW + (n % PW);
  uint4_t kr[QD / 16];
  {
    const int t = min(tk, span_count - 1);
    const int slot = ring_slot(t);
    const uint4_t *row =
        reinterpret_cast<const uint4_t *>(a.key_store + (size_t)slot * a.kv_width + kv_off + QD * g);
#pragma unroll
    for (int q = 0; q < QD / 16; ++q) kr[q] = __builtin_nontemporal_load(row + q);
  }
  // value rows: row (lane / LPR) + RPI*i of the chunk, bytes of dims
  // wave*DS + 16*(lane % LPR) .. + 15
  uint4_t vr[VL];
#pragma unroll
  for (int i = 0; i < VL; ++i) {
    const int t = min(c0 + lane / LPR + RPI * i, span_count - 1);
    const int slot = ring_slot(t);
    vr[i] = __builtin_nontemporal_load(reinterpret_cast<const uint4_t *>(
        a.value_store + (size_t)slot * a.kv_width + kv_off + wave * DS + 16 * (lane % LPR)));
  }

  if (PREP) {
    // Each head's items are 32 (HEAD 256) or 64 (HEAD 512) consecutive
    // threads; the pair (j, j + HALF) of a dim sits HALF / 8 items apart.
#pragma unroll
    for (int i = 0; i < kQItems; ++i) {
      const int item = tid + 256 * i;
      const int d0 = 8 * (item % kHeadItems);
      double ss = 0.0;
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += (double)qf[i][e] * (double)qf[i][e];
#pragma unroll
      for (int off = kHeadItems / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
      const float shrink = rms_shrink(ss, HEAD, a.eps);
      float own[8], other[8];
      const float4_t g0 = qgain[i][0], g1 = qgain[i][1];
      const float gg[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        own[e] = qf[i][e] * shrink;
        own[e] = own[e] * gg[e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) other[e] = __shfl_xor(own[e], kHeadItems / 2);
      const bool low = d0 < HALF;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float c = qturn[i][e >> 1][2 * (e & 1)];
        const float sn = qturn[i][e >> 1][2 * (e & 1) + 1];
        qf[i][e] = low ? own[e] * c - other[e] * sn : own[e] * c + other[e] * sn;
      }
    }
  }

  // query operands, x = hi + lo in binary16
#pragma unroll
  for (int i = 0; i < kQItems; ++i) {
    half8_t hi8, lo8;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const _Float16 hi = (_Float16)qf[i][e];
      hi8[e] = hi;
      lo8[e] = (_Float16)(qf[i][e] - (float)hi);
    }
    const int item = tid + 256 * i;
    qs[0][item / (HEAD / 8)][item % (HEAD / 8)] = hi8;
    qs[1][item / (HEAD / 8)][item % (HEAD / 8)] = lo8;
  }
  __syncthreads();

  // ---- scores of the wave's PW positions for the 8 heads, all dims
  float sc[4];
  float m_w[4];
  {
    float4_t sacc = float4_t{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const half8_t qa = qs[n >> 3][n & 7][QD * g / 8 + s];
      const uint4_t w = kr[s >> 1];
      const half8_t kb = (s & 1) ? decode8<FMT>(w[2], w[3]) : decode8<FMT>(w[0], w[1]);
      sacc = __builtin_amdgcn_mfma_f32_16x16x32_f16(qa, kb, sacc, 0, 0, 0);
    }
    const bool valid = n < PW && tk < span_count;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = xsum32(sacc[r]);
      sc[r] = valid ? v * a.key_scale : -INFINITY;
      m_w[r] = row16_max(sc[r]);
    }
  }
  // probabilities against the wave's peak, and the wave's sums
  {
    float l_w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float p = m_w[r] != -INFINITY && sc[r] != -INFINITY ? __expf(sc[r] - m_w[r]) : 0.0f;
      l_w[r] = row16_sum(p);
      if (g < 2 && n < PW) ps[4 * g + r][wave * PW + n] = p;
    }
    if (g < 2 && n == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        wm[wave][4 * g + r] = m_w[r];
        wl[wave][4 * g + r] = l_w[r];
      }
    }
  }
  // the wave's value slice into its own LDS rows
  {
    uint8_t *vw = vs[wave];
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      uint2_t *dst = reinterpret_cast<uint2_t *>(vw + (lane / LPR + RPI * i) * VP + 16 * (lane % LPR));
      dst[0] = uint2_t{vr[i][0], vr[i][1]};
      dst[1] = uint2_t{vr[i][2], vr[i][3]};
    }
  }
  __syncthreads();

  // ---- blend of the wave's dims over the chunk's positions.  A = the
  // probabilities (row n: head n & 7, hi part for n < 8, lo part otherwise;
  // k = positions 8g .. 8g + 7 of the k-step), each scaled by e^(m_w - M),
  // M the chunk's peak of the head.
  const int hh = n & 7;
  float M = wm[0][hh];
#pragma unroll
  for (int w = 1; w < W; ++w) M = fmaxf(M, wm[w][hh]);
  float4_t o[4 * QUADS];
#pragma unroll
  for (int t = 0; t < 4 * QUADS; ++t) o[t] = float4_t{0, 0, 0, 0};
  const uint8_t *vw = vs[wave];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int p0 = 32 * ks + 8 * g;  // the lane's first position of the k-step
    const float mw = wm[p0 / PW][hh];
    const float f = mw != -INFINITY ? __expf(mw - M) : 0.0f;
    half8_t pa;
    {
      const float *src = &ps[hh][p0];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = src[e] * f;
        const _Float16 hi = (_Float16)v;
        pa[e] = n >= 8 ? (_Float16)(v - (float)hi) : hi;
      }
    }
#pragma unroll
    for (int qd = 0; qd < QUADS; ++qd) {
      uint32_t dw[8];
#pragma unroll
      for (int e = 0; e < 8; ++e)
        dw[e] = *reinterpret_cast<const uint32_t *>(vw + (p0 + e) * VP + 64 * qd + 4 * n);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        uint32_t w[4];
        const uint32_t sel = 0x0C000C00u | ((uint32_t)(4 + t) << 16) | (uint32_t)t;
#pragma unroll
        for (int pr = 0; pr < 4; ++pr)
          w[pr] = decode_pair<FMT>(__builtin_amdgcn_perm(dw[2 * pr + 1], dw[2 * pr], sel));
        o[4 * qd + t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa, __builtin_bit_cast(half8_t, w),
                                                               o[4 * qd + t], 0, 0, 0);
      }
    }
  }
  // hi + lo rows; lanes g < 2 hold head 4g + r, dims wave*DS + 64qd + 4n + t
#pragma unroll
  for (int t = 0; t < 4 * QUADS; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) o[t][r] = xsum32(o[t][r]);
  if (g >= 2) return;
  // the waves' peaks and sums of heads 4g .. 4g + 3, read at once
  float4_t pk[W], tl[W];
#pragma unroll
  for (int w = 0; w < W; ++w) {
    pk[w] = *reinterpret_cast<const float4_t *>(&wm[w][4 * g]);
    tl[w] = *reinterpret_cast<const float4_t *>(&wl[w][4 * g]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int h = 4 * g + r;
    float Mh = pk[0][r];
#pragma unroll
    for (int w = 1; w < W; ++w) Mh = fmaxf(Mh, pk[w][r]);
    float L = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float e = pk[w][r] != -INFINITY ? __expf(pk[w][r] - Mh) : 0.0f;
      L += tl[w][r] * e;
    }
    float *dst;
    float mul;
    if (a.final_out) {
      dst = a.final_out + (size_t)lane_id * a.q_stride + (size_t)(head0 + h) * HEAD + wave * DS + 4 * n;
      mul = L > 0.0f ? a.value_scale * (1.0f / L) : 0.0f;
    } else {
      dst = a.part_out + ((size_t)pc * a.head_count + head0 + h) * HEAD + wave * DS + 4 * n;
      mul = a.value_scale;
      if (wave == 0 && n == 0) {
        a.part_peak[(size_t)pc * a.head_count + head0 + h] = Mh;
        a.part_total[(size_t)pc * a.head_count + head0 + h] = L;
      }
    }
#pragma unroll
    for (int qd = 0; qd < QUADS; ++qd)
      *reinterpret_cast<float4_t *>(dst + 64 * qd) =
          float4_t{o[4 * qd][r] * mul, o[4 * qd + 1][r] * mul, o[4 * qd + 2][r] * mul, o[4 * qd + 3][r] * mul};
  }
}

// ---- tiles of lanes ----------------------------------------------------------
//
// A launch of many lanes (a prompt's pass, a block) takes tiles of 2 RB lanes:
// their 8 query heads are the 16 RB rows of the MFMA tiles, so a key or value
// byte is read and decoded once for all of them (a chunk workgroup decodes
// every byte for one lane's 8, and its 16 MFMA rows hold each head's two
// terms).  A workgroup of a wave for every 64 dims walks the chunks of 64
// positions of the tile's span (its first lane's first position to its last
// lane's own), or of one segment of it (blockIdx.z).  Both products are split
// among the waves by dims: wave w takes dims 64 w .. of the scores, whose
// partial sums the waves exchange through LDS, and the same dims of the blend.
// So a wave holds its slice of the queries (both terms) and of the blend in
// registers for the whole walk, and the LDS DMA brings its key and value bytes
// into rows only it reads, the keys a chunk ahead: two barriers a chunk.
//
// What bounds it: a chunk's chain between the two barriers (decode, products,
// the exchanged sums, the exponentials; 6200 cycles a chunk of 512-dim heads at
// 32 rows, 2000 of them products on each SIMD).  At 2047 lanes, us, against one
// workgroup a lane: 2048 positions of 512-dim heads 450 -> 99 (69 GFLOP of
// products, two terms each: 695 TFLOP/s), a 512 window of 256-dim heads 104 -> 34;
// 511 lanes 57 -> 22.  Slower: four waves of 128 dims, two workgroups a CU (9%: a
// chunk's chain is 8800 cycles, and the longest tile's chunks bound the launch);
// the keys in registers instead of LDS (41%: spills).
//
// Per chunk: scores S = q_lo . K^T + q_hi . K^T (the waves' sums added in wave
// order, in powers of two: log2 e is in the key scale), probabilities p = 2^(S -
// base) to LDS as two binary16 terms, and total and blend = blend 2^(old base -
// base) + (p_lo + p_hi) . V, each chunk's products formed from zero.  A row's base
// is the chunk's peak rounded down, so p's largest is in [1, 2), its two terms
// lose no more than half of 2^-24 of that, and every scaling is exact.  Against
// the walk's running peak, the weights far below an early position's fall under
// binary16's range: one position 18 (base e) above 1000-1900 others, its own value
// zero, left the blend 12% (256 dims) and 40% (512) off, here 4.4% and 4.9%, the
// share of the chunk that holds it.  No base is more than 58 under the largest
// one, so the scaled sums stay in fp32's range.  Off the 64-bit blend at 64-515
// lanes, scores of deviation 1, 6 and 30: 1.6e-7, 4.5e-7, 9.4e-7 (chunk workgroups
// 2.2e-7, 7.8e-7, 1.6e-6).  Positions a lane does not see have probability zero in
// its rows.
typedef __attribute__((address_space(3))) void attend_lds_t;
typedef __attribute__((address_space(1))) const void attend_global_t;

__device__ __forceinline__ void lds_barrier() {
  // LDS only: the key bytes requested ahead stay in flight
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// A buffer over the rows at a uniform address: its loads take the address in
// scalar registers and a 32-bit lane offset (as pointers, the compiler keeps
// 64-bit lane addresses through the loop and spills).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t uniform_rows(const uint8_t *rows) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(rows), 0, 0xFFFFFFFF, 0x00020000);
}

// LDS of a tile workgroup, in bytes: its waves' key rows (and then their
// partial scores, rows of 68 floats), the probabilities' two terms (rows of 72
// halves), a float a row, the waves' value rows.
template <int HEAD, int RB>
struct TileLds {
  static constexpr int W = HEAD / 64;
  static constexpr int KEYS = 64 * 64, SCORES = 16 * RB * 68 * 4;
  static constexpr int KR = KEYS > SCORES ? KEYS : SCORES;
  static constexpr int P = W * KR;
  static constexpr int KEEP = P + 2 * 16 * RB * 72 * 2;
  static constexpr int V = KEEP + 16 * RB * 4;
  static constexpr int SIZE = V + 64 * HEAD;
};

template <int HEAD, int FMT, int RB, bool QVEC>
__global__ __launch_bounds__(HEAD, 2) void attend_tile_kernel(AttendArgs a) {
  constexpr int LT = 2 * RB;          // lanes a tile
  constexpr int ROWS = 16 * RB;       // (lane, head) rows
  constexpr int C = 64;               // positions a chunk
  constexpr int W = HEAD / 64;        // waves: a thread a dim
  constexpr int DS = 64;              // dims a wave holds
  constexpr int S = DS / 32;          // k-steps of its scores
  constexpr int QD = DS / 4;          // dims (and key bytes a position) one lane group reads
  constexpr int LPR = DS / 16;        // 16-byte chunks of a staged value row
  constexpr int RPI = 64 / LPR;       // value rows one DMA instruction covers
  constexpr int VL = C / RPI;         // DMA instructions of a chunk's values
  constexpr int RP = C + 4;           // score row pitch in floats
  constexpr int PP = C + 8;           // probability row pitch in halves
  constexpr int TPR = HEAD / ROWS < 16 ? HEAD / ROWS : 16;  // threads a row in the softmax
  constexpr int PPT = C / TPR;        // positions a thread

  // one array, laid out by hand: between arrays the compiler would wait for
  // the DMA into one before any read of another
  using F = TileLds<HEAD, RB>;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  _Float16 *ph = reinterpret_cast<_Float16 *>(lds + F::P), *pl = ph + ROWS * PP;
  float *keep_s = reinterpret_cast<float *>(lds + F::KEEP);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4;
  const int n = lane & 15;
  const int kv = blockIdx.y;
  const int head0 = kv * kAttendGroup;
  const size_t kv_off = (size_t)kv * HEAD;
  // Longest tiles first, as a CU frees.  Where two workgroups share a CU and
  // all fit at once (256-dim heads), the second half starts with the shortest,
  // so a causal launch's long tiles each meet a short one on their CU.
  const int tiles = gridDim.x, half = W == 4 && tiles <= 512 ? (tiles + 1) / 2 : tiles;
  const int tile = (int)blockIdx.x < half ? tiles - 1 - (int)blockIdx.x : (int)blockIdx.x - half;
  const int l0 = tile * LT;
  const int ln = min(LT, a.lanes - l0);
  const int pos0 = __builtin_amdgcn_readfirstlane(a.place_dev ? *a.place_dev : a.place0) + l0;
  const int start = a.window > 0 ? max(0, pos0 + 1 - a.window) : 0;
  const int span = pos0 + ln - start;  // of the tile
  const int chunks = (span + C - 1) / C;
  const int per = (chunks + (int)gridDim.z - 1) / (int)gridDim.z;
  const int seg = blockIdx.z;
  const int c_first = seg * per, c_end = min(chunks, c_first + per);
  const bool split = gridDim.z > 1;

  // the softmax's row of this thread, its lane's visible positions (relative
  // to start), its largest base, its base and its running total
  const int row = min(tid / TPR, ROWS - 1);
  const int li = min(row / kAttendGroup, ln - 1);
  const int see_end = pos0 + li - start;  // inclusive
  const int see_first = a.window > 0 ? max(0, pos0 + li + 1 - a.window) - start : 0;
  float top = -INFINITY, run_m = -INFINITY, run_l = 0.0f;

  const int ring0 = start % a.cache_span;
  // t < span < 2 cache_span (the host takes this form past 64 visible positions)
  auto ring_slot = [&](int t) {
    int slot = ring0 + t;
    slot = slot >= a.cache_span ? slot - a.cache_span : slot;
    return slot >= a.cache_span ? slot - a.cache_span : slot;
  };
  // A whole chunk in consecutive slots (nearly all are) is read at lane
  // offsets from one uniform address; else each row finds its own slot.
  // Key row p holds its 16-byte chunk ch at chunk ch ^ (p / 4) % 4, so the 16
  // rows a score read spans lie in distinct banks.
  uint8_t *kw = lds + F::KR * wave;
  const int k_row = lane / LPR;
  const int k_chunk = 16 * ((lane % 4) ^ (lane >> 4));
  const uint32_t k_lane = (uint32_t)(k_row * a.kv_width + k_chunk);
  auto load_keys = [&](int c) {
    const int slot0 = ring_slot(c * C);
    const uint8_t *keys = a.key_store + kv_off + wave * DS;
    if (c * C + C <= span && slot0 + C <= a.cache_span) {
      const auto src = uniform_rows(keys + (size_t)slot0 * a.kv_width);
#pragma unroll
      for (int i = 0; i < VL; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (attend_lds_t *)(kw + 1024 * i), 16, k_lane,
                                                 RPI * i * a.kv_width, 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < VL; ++i) {
        const int t = min(c * C + RPI * i + k_row, span - 1);
        __builtin_amdgcn_global_load_lds(
            (attend_global_t *)(keys + (size_t)ring_slot(t) * a.kv_width + k_chunk),
            (attend_lds_t *)(kw + 1024 * i), 16, 0, 0);
      }
    }
  };
  // Value row p goes to row slot (p & ~3) + (p + p / 8) % 4: a blend read takes
  // 64 bytes of rows p, p + 8, p + 16 and p + 24, which so lie in four distinct
  // quarters of the banks.  Instruction i fills slots RPI i + lane / LPR; v_row
  // is the lane's row in an even and an odd one.
  uint8_t *vw = lds + F::V + C * DS * wave;
  int v_row[2];
  uint32_t v_lane[2];
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    v_row[o] = ((lane / LPR) & ~3) | ((lane / LPR - 2 * o - (lane >> 5)) & 3);
    v_lane[o] = (uint32_t)(v_row[o] * a.kv_width + 16 * (lane % LPR));
  }
  auto load_values = [&](int c) {
    const int slot0 = ring_slot(c * C);
    const uint8_t *values = a.value_store + kv_off + wave * DS;
    if (c * C + C <= span && slot0 + C <= a.cache_span) {
      const auto src = uniform_rows(values + (size_t)slot0 * a.kv_width);
#pragma unroll
      for (int i = 0; i < VL; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (attend_lds_t *)(vw + 1024 * i), 16,
                                                 v_lane[i & 1], RPI * i * a.kv_width, 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < VL; ++i) {
        const int t = min(c * C + RPI * i + v_row[i & 1], span - 1);
        __builtin_amdgcn_global_load_lds(
            (attend_global_t *)(values + (size_t)ring_slot(t) * a.kv_width + 16 * (lane % LPR)),
            (attend_lds_t *)(vw + 1024 * i), 16, 0, 0);
      }
    }
  };
  // the lane's blend reads of its eight rows p0 .. p0 + 7 (p0 = 32 ks + 8 g)
  const uint8_t *v_read[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v_read[e] = vw + 512 * g + 64 * ((e + g) & 3) + 4 * n;
  if (c_first < c_end) load_keys(c_first);

  // the wave's slice of the queries, x = hi + lo: row 16 rb + n is lane 2 rb +
  // n / 8, head n % 8; k-step s of lane group g is dims QD g + 8 s .. + 7
  half8_t qh[RB][S], ql[RB][S];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int lq = l0 + min(2 * rb + (n >> 3), ln - 1);
    const float *q = a.query + (size_t)lq * a.q_stride + (size_t)(head0 + (n & 7)) * HEAD + wave * DS + QD * g;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      float x[8];
      if (QVEC) {
        const float4_t u = *reinterpret_cast<const float4_t *>(q + 8 * s);
        const float4_t v = *reinterpret_cast<const float4_t *>(q + 8 * s + 4);
        x[0] = u.x; x[1] = u.y; x[2] = u.z; x[3] = u.w;
        x[4] = v.x; x[5] = v.y; x[6] = v.z; x[7] = v.w;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = q[8 * s + e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const _Float16 hi = (_Float16)x[e];
        qh[rb][s][e] = hi;
        ql[rb][s][e] = (_Float16)(x[e] - (float)hi);
      }
    }
  }

  // the blend: rows 16 rb + 4 g + r, dims wave DS + 4 n + t
  float4_t out[RB][4];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int t = 0; t < 4; ++t) out[rb][t] = float4_t{0, 0, 0, 0};

  for (int c = c_first; c < c_end; ++c) {
    asm volatile("" ::: "memory");
    load_values(c);  // the chunk before's reads of these rows have been multiplied
    __builtin_amdgcn_s_waitcnt(0xF70 | VL);  // the keys, requested before, have landed
    asm volatile("" ::: "memory");
    // scores over the wave's dims
    float4_t sc[RB][4];
#pragma unroll
    for (int pb = 0; pb < 4; ++pb) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) sc[rb][pb] = float4_t{0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const uint4_t w = *reinterpret_cast<const uint4_t *>(kw + (16 * pb + n) * DS + 16 * (g ^ (n >> 2)));
        const half8_t kb = (s & 1) ? decode8<FMT>(w[2], w[3]) : decode8<FMT>(w[0], w[1]);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          sc[rb][pb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ql[rb][s], kb, sc[rb][pb], 0, 0, 0);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          sc[rb][pb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(qh[rb][s], kb, sc[rb][pb], 0, 0, 0);
      }
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int pb = 0; pb < 4; ++pb)
#pragma unroll
        for (int r = 0; r < 4; ++r) reinterpret_cast<float *>(kw)[(16 * rb + 4 * g + r) * RP + 16 * pb + n] = sc[rb][pb][r];
    lds_barrier();
    // the row's scores of this thread, its peak and total, its probabilities
    if (ROWS * TPR == HEAD || tid < ROWS * TPR) {
      const int p0 = PPT * (tid % TPR);
      float raw[PPT], v[PPT];
#pragma unroll
      for (int e = 0; e < PPT; e += 4) {
        float4_t x[W];
#pragma unroll
        for (int w = 0; w < W; ++w) x[w] = reinterpret_cast<const float4_t *>(lds + F::KR * w)[(row * RP + p0 + e) / 4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int w = W / 2; w > 0; w >>= 1)
#pragma unroll
            for (int j = 0; j < w; ++j) x[j][i] += x[j + w][i];
          raw[e + i] = x[0][i];
          v[e + i] = x[0][i] * a.key_scale;
        }
      }
      // uniform in a wave: some of its rows do not see all of the chunk
      const int t0 = c * C;
      if (t0 < see_first || t0 + C - 1 > see_end) {
#pragma unroll
        for (int e = 0; e < PPT; ++e) {
          const int t = t0 + p0 + e;
          if (t < see_first || t > see_end) v[e] = -INFINITY;
        }
      }
      float peak = v[0];
#pragma unroll
      for (int e = 1; e < PPT; ++e) peak = fmaxf(peak, v[e]);
      peak = fmaxf(peak, dpp_move<0xB1>(peak));
      peak = fmaxf(peak, dpp_move<0x4E>(peak));
      if (TPR >= 8) peak = fmaxf(peak, dpp_move<0x141>(peak));
      if (TPR >= 16) peak = fmaxf(peak, dpp_move<0x140>(peak));
      const float low = floorf(peak);
      top = fmaxf(top, low);
      const float m = fmaxf(low, top - 58.0f);
      const float keep = run_m != -INFINITY ? __builtin_amdgcn_exp2f(run_m - m) : 0.0f;
      float total = 0.0f;
      _Float16 hi[PPT], lo[PPT];
#pragma unroll
      for (int e = 0; e < PPT; ++e) {
        // the score's scale and its distance from the base in one rounding
        const float p = v[e] != -INFINITY ? __builtin_amdgcn_exp2f(__builtin_fmaf(raw[e], a.key_scale, -m)) : 0.0f;
        total += p;
        hi[e] = (_Float16)p;
        lo[e] = (_Float16)(p - (float)hi[e]);
      }
      total += dpp_move<0xB1>(total);
      total += dpp_move<0x4E>(total);
      if (TPR >= 8) total += dpp_move<0x141>(total);
      if (TPR >= 16) total += dpp_move<0x140>(total);
      run_l = run_l * keep + total;
      run_m = m;
      __builtin_memcpy(__builtin_assume_aligned(&ph[row * PP + p0], 8), hi, sizeof(hi));
      __builtin_memcpy(__builtin_assume_aligned(&pl[row * PP + p0], 8), lo, sizeof(lo));
      if (tid % TPR == 0) keep_s[row] = keep;
    }
    // the wave's values have landed: their reads go out before the barrier
    __builtin_amdgcn_s_waitcnt(0xF70);
    asm volatile("" ::: "memory");
    uint32_t dw[C / 32][8];
#pragma unroll
    for (int ks = 0; ks < C / 32; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        dw[ks][e] = *reinterpret_cast<const uint32_t *>(v_read[e & 3] + 2048 * ks + 256 * (e >> 2));
    lds_barrier();
    if (c + 1 < c_end) load_keys(c + 1);  // every wave has read the scores that lay there
    // the blend over the wave's dims
    float4_t o[RB][4];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int t = 0; t < 4; ++t) o[rb][t] = float4_t{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < C / 32; ++ks) {
      half8_t pa[RB][2];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        pa[rb][0] = *reinterpret_cast<const half8_t *>(&ph[(16 * rb + n) * PP + 32 * ks + 8 * g]);
        pa[rb][1] = *reinterpret_cast<const half8_t *>(&pl[(16 * rb + n) * PP + 32 * ks + 8 * g]);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        uint32_t w[4];
        const uint32_t sel = 0x0C000C00u | ((uint32_t)(4 + t) << 16) | (uint32_t)t;
#pragma unroll
        for (int pr = 0; pr < 4; ++pr)
          w[pr] = decode_pair<FMT>(__builtin_amdgcn_perm(dw[ks][2 * pr + 1], dw[ks][2 * pr], sel));
        const half8_t vb = __builtin_bit_cast(half8_t, w);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          o[rb][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[rb][1], vb, o[rb][t], 0, 0, 0);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          o[rb][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[rb][0], vb, o[rb][t], 0, 0, 0);
      }
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const float4_t keep = *reinterpret_cast<const float4_t *>(&keep_s[16 * rb + 4 * g]);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[rb][t][r] = __builtin_fmaf(out[rb][t][r], keep[r], o[rb][t][r]);
    }
  }

  // the rows' totals to every wave; with segments the partial, else the blend
  lds_barrier();
  if (tid % TPR == 0 && tid < ROWS * TPR) {
    keep_s[row] = run_l;
    if (split && row / kAttendGroup < ln) {
      const size_t at = ((size_t)(l0 + row / kAttendGroup) * gridDim.z + seg) * a.head_count + head0 + (row & 7);
      a.part_peak[at] = run_m;
      a.part_total[at] = run_l;
    }
  }
  lds_barrier();
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * rb + 4 * g + r;
      const int l = m / kAttendGroup, h = head0 + (m & 7);
      if (l >= ln) continue;
      const float total = keep_s[m];
      const float mul = split ? a.value_scale : total > 0.0f ? a.value_scale * (1.0f / total) : 0.0f;
      float *dst = (split ? a.part_out + (((size_t)(l0 + l) * gridDim.z + seg) * a.head_count + h) * HEAD
                          : a.final_out + (size_t)(l0 + l) * a.q_stride + (size_t)h * HEAD) + wave * DS + 4 * n;
      const float4_t o4 = {out[rb][0][r] * mul, out[rb][1][r] * mul, out[rb][2][r] * mul, out[rb][3][r] * mul};
      if (QVEC || split) {
        *reinterpret_cast<float4_t *>(dst) = o4;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e] = o4[e];
      }
    }
}

template <bool TWO>
__device__ __forceinline__ float fold_power(float x) {
  return TWO ? __builtin_amdgcn_exp2f(x) : __expf(x);
}

// Folds chunk partials in one memory round trip.  A workgroup per (head, lane,
// DIMS dims) of 256 threads: thread (d, s) loads, for up to PER chunks
// c = s, s + 256/DIMS, ..., its dim's partial and the chunk's peak and total
// together; the slices' peaks meet in LDS (the head's peak M), each thread
// weights its chunks by e^(peak_c - M), and the slices' sums meet in LDS in a
// fixed order.  Spans of more chunks than one pass holds take further passes,
// each rescaled to the running peak.  TWO: the peaks are powers of two (a tile's
// segments), not of e.
template <int DIMS, int PER, bool TWO>
__global__ __launch_bounds__(256) void attend_fold_kernel(const float *part_out_all,
                                                          const float *part_peak_all,
                                                          const float *part_total_all,
                                                          int chunk_slots, int chunk, int place0,
                                                          const int *place_dev, int window,
                                                          int extra, int head_count, int head_size,
                                                          float *blend_all, int o_stride) {
  constexpr int SL = 256 / DIMS;
  __shared__ float red_m[SL];
  __shared__ float red_a[SL][DIMS];
  __shared__ float red_l[SL];
  const int h = blockIdx.x, lane_id = blockIdx.y, tid = threadIdx.x;
  const int d = tid % DIMS, sl = tid / DIMS;
  const int pos = (place_dev ? *place_dev : place0) + lane_id;
  const int span = window > 0 ? min(pos + 1, window) : pos + 1;
  // extra: the block's new positions up to the lane's own have a partial of
  // their own, after the chunks of the positions before the block
  const int fresh = extra ? lane_id + 1 : 0;
  // chunk 0: every lane fills its slots, those of no position with a zero blend
  const int chunks = chunk ? (span - fresh + chunk - 1) / chunk + (extra ? 1 : 0) : chunk_slots;
  const size_t base = (size_t)lane_id * chunk_slots;
  const size_t step = (size_t)head_count * head_size;
  const float *pout = part_out_all + base * step + (size_t)h * head_size + blockIdx.z * DIMS + d;
  const float *ppk = part_peak_all + base * head_count + h;
  const float *ptt = part_total_all + base * head_count + h;
  float run_m = -INFINITY, acc = 0.0f, tot = 0.0f;
  for (int c0 = 0; c0 < chunks; c0 += SL * PER) {
    float v[PER], m[PER], l[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int c = min(c0 + sl + SL * u, chunks - 1);
      v[u] = pout[(size_t)c * step];
      m[u] = ppk[(size_t)c * head_count];
      l[u] = ptt[(size_t)c * head_count];
    }
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < PER; ++u)
      if (c0 + sl + SL * u < chunks) mx = fmaxf(mx, m[u]);
    __syncthreads();  // red_m of the previous pass read by every thread
    if (d == 0) red_m[sl] = mx;
    __syncthreads();
    float M = run_m;
#pragma unroll
    for (int i = 0; i < SL; ++i) M = fmaxf(M, red_m[i]);
    if (M != -INFINITY && run_m != -INFINITY && M != run_m) {
      const float f = fold_power<TWO>(run_m - M);
      acc *= f;
      tot *= f;
    }
    run_m = M;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const bool in = c0 + sl + SL * u < chunks && m[u] != -INFINITY;
      const float w = in ? fold_power<TWO>(m[u] - M) : 0.0f;
      acc += w * v[u];
      tot += w * l[u];
    }
  }
  red_a[sl][d] = acc;
  if (d == 0) red_l[sl] = tot;
  __syncthreads();
  if (sl == 0) {
    float A = 0.0f, T = 0.0f;
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      A += red_a[i][d];
      T += red_l[i];
    }
    blend_all[(size_t)lane_id * o_stride + (size_t)h * head_size + blockIdx.z * DIMS + d] =
        T == 0.0f ? 0.0f : A * (1.0f / T);  // NaN: a lane whose scores are
  }
}

}  // namespace igl

using namespace igl;

static int attend_max_span(int place0, int window, int lanes) {
  const int last = place0 + lanes;  // span of the last lane when unwindowed
  return window > 0 ? (last < window ? last : window) : last;
}

static int attend_chunk(int place0, int window, int lanes) {
  if (lanes >= kAttendWideLanes) return 64;
  return attend_max_span(place0, window, lanes) <= kAttendShortSpan ? 32 : 64;
}

static int attend_blocks(int place0, int window, int lanes) {
  const int chunk = attend_chunk(place0, window, lanes);
  return (attend_max_span(place0, window, lanes) + chunk - 1) / chunk;
}

// Which launches take tiles of lanes (attend_tile_kernel), and their shape.
//
// Spans past 64 positions (up to there one chunk workgroup a lane writes the
// blend), and
//   * from 64 lanes: always;
//   * below: two lanes and more of 512-dim heads; of 256-dim heads where the
//     chunk form would take 512 workgroups and more.  Replayed, us, chunk
//     workgroups and fold -> tiles: 512 dims, 2 lanes at 300 positions 9.9 -> 8.6
//     (16000: 22.5 -> 15.5), 16 lanes 11.2 -> 9.3, 63 lanes 23.3 -> 14.4, 32
//     lanes at 16000 216 -> 40; 256 dims, 63 lanes of a 512 window 15.8 -> 11.9, 5
//     lanes at 16000 26.7 -> 14.9, but 4 lanes of the window 7.7 against 7.9, 16
//     lanes 8.5 against 8.9, 2 lanes at 16000 (502 chunk workgroups) 12.8
//     against 13.2.
// Tiles of two lanes up to 512 of them, of four beyond (us in twos and in fours:
// 1000 lanes of 512 dims 46.9, 49.9; 1100 54.4, 55.4; 1500 82.0, 72.3; 2047 127.8,
// 101.5; 2047 of a 512 window of 256 dims 41.0, 36.7).
//
// Few tiles are cut into segments of their chunks, folded by a second launch:
// as many as fill 256 workgroups, 512 (512 dims) or 1024 (256 dims) where a
// segment would still be more than eight chunks long, 64 at most.  100 lanes at
// 2000 positions, 256 dims: unsplit 55.7 us, five segments 22; 300 lanes of a
// 512 window: unsplit 19.0, two 22.5; 32 lanes at 16000, 512 dims: 16 segments
// 44.2, 32 40.4, 64 45.6.  The partials stay within what the same call's chunk
// form takes below 64 lanes; from there within what 48 lanes' chunk form would
// take (the engine's workspace holds 63 lanes') and IGL_ATTEND_FIXED_FLOATS.
struct TilePlan {
  int rb;        // lanes a tile / 2; 0: not this form
  int segments;
};

static TilePlan attend_tile_plan(int place0, int window, int lanes, int head_count, int head_size) {
  const TilePlan none = {0, 1};
  if (lanes < 2) return none;
  const int span = attend_max_span(place0, window, lanes);
  const int kv_count = head_count / kAttendGroup;
  const bool wide = lanes >= kAttendWideLanes;
  const long blocks = (span + (span <= kAttendShortSpan ? 31 : 63)) / (span <= kAttendShortSpan ? 32 : 64);
  if (span <= 64) return none;
  if (!wide && head_size == 256 && (long)lanes * kv_count * blocks < 512) return none;
  const int rb = (long)((lanes + 1) / 2) * kv_count <= 512 ? 1 : 2;
  const long tiles = (long)((lanes + 2 * rb - 1) / (2 * rb)) * kv_count;
  const long chunks = (span + 2 * rb - 1 + 63) / 64;  // of a tile, at most
  long s = 256 / tiles;
  if (s < 1) s = 1;
  if (chunks > 8 * s) s = (head_size == 256 ? 1024 : 512) / tiles;
  if (wide) {
    const long fixed = (long)IGL_ATTEND_FIXED_FLOATS / ((long)lanes * head_count * (head_size + 2));
    if (s > 48 * blocks / lanes) s = 48 * blocks / lanes;
    if (s > fixed) s = fixed;
  }
  if (s > 64) s = 64;
  if (s > blocks) s = blocks;
  if (s > chunks) s = chunks;
  if (s < 1) s = 1;
  const long per = (chunks + s - 1) / s;
  return TilePlan{rb, (int)((chunks + per - 1) / per)};
}

template <int HEAD, int FMT, int C>
static void attend_launch(const AttendArgs &a, dim3 grid, bool qvec, hipStream_t stream) {
  if (qvec)
    hipLaunchKernelGGL((attend_split_kernel<HEAD, FMT, C, true, false>), grid, dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((attend_split_kernel<HEAD, FMT, C, false, false>), grid, dim3(256), 0, stream, a);
}

template <int HEAD, int FMT, int RB, bool QVEC>
static hipError_t attend_launch_tiles(const AttendArgs &a, int kv_count, int segments, hipStream_t stream) {
  constexpr int size = TileLds<HEAD, RB>::SIZE;
  static bool granted = false;  // the dynamic LDS a kernel asks for is granted once
  if (!granted) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&attend_tile_kernel<HEAD, FMT, RB, QVEC>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, size);
    if (e != hipSuccess) return e;
    granted = true;
  }
  const dim3 grid((a.lanes + 2 * RB - 1) / (2 * RB), kv_count, segments);
  hipLaunchKernelGGL((attend_tile_kernel<HEAD, FMT, RB, QVEC>), grid, dim3(HEAD), (size_t)size, stream, a);
  return hipGetLastError();
}

template <int HEAD, int FMT>
static hipError_t attend_launch_tile(const AttendArgs &a, const TilePlan &p, int kv_count, bool qvec,
                                     hipStream_t stream) {
  if (p.rb == 1)
    return qvec ? attend_launch_tiles<HEAD, FMT, 1, true>(a, kv_count, p.segments, stream)
                : attend_launch_tiles<HEAD, FMT, 1, false>(a, kv_count, p.segments, stream);
  return qvec ? attend_launch_tiles<HEAD, FMT, 2, true>(a, kv_count, p.segments, stream)
              : attend_launch_tiles<HEAD, FMT, 2, false>(a, kv_count, p.segments, stream);
}

template <int HEAD, int FMT>
static void attend_launch_chunk(const AttendArgs &a, dim3 grid, int chunk, bool qvec, hipStream_t stream) {
  if (chunk == 32)
    attend_launch<HEAD, FMT, 32>(a, grid, qvec, stream);
  else
    attend_launch<HEAD, FMT, 64>(a, grid, qvec, stream);
}

static hipError_t attend_fold(const AttendArgs &a, int chunks, int chunk, int place0,
                              const int *place_dev, int window, int lanes, int head_size,
                              float *blend_out, hipStream_t stream, int extra = 0);

// `lanes` query lanes at positions place0 .. place0 + lanes - 1, each seeing
// the last `window` positions up to its own (0: every position from 0).  Lane
// l's query and output are `q_stride` floats after lane l - 1's.  With
// `place_dev`, lane 0's position is read from device memory when the kernels
// run and `place0` is only its upper bound, which sizes the grid (a launch
// that a graph replays at every step).
extern "C" hipError_t igl_launch_attend(const uint8_t *key_store, const uint8_t *value_store,
                                        int fmt, float key_scale, float value_scale,
                                        int cache_span, int kv_width, int kv_count,
                                        int group_share, int head_size, const float *query,
                                        int q_stride, int place0, const int *place_dev,
                                        int window, int lanes, float score_scale,
                                        float *blend_out, float *work, hipStream_t stream) {
  AttendArgs a;
  const int chunk = attend_chunk(place0, window, lanes);
  const int chunks = attend_blocks(place0, window, lanes);  // workgroups a lane
  const int head_count = kv_count * group_share;
  if (group_share != kAttendGroup || lanes < 1) return hipErrorInvalidValue;
  a.key_store = key_store;
  a.value_store = value_store;
  a.kv_width = kv_width;
  a.cache_span = cache_span;
  a.place0 = place0;
  a.place_dev = place_dev;
  a.window = window;
  a.lanes = lanes;
  a.chunks = chunks;
  a.final_out = chunks == 1 ? blend_out : nullptr;
  a.q_stride = q_stride;
  a.query = query;
  // e4m3 decodes to real8 / 256; the 256 goes back in with the scale.
  const float unit = fmt == 0 ? 256.0f : 1.0f;
  a.key_scale = key_scale * unit * score_scale;
  a.value_scale = value_scale * unit;
  a.head_count = head_count;
  const size_t slots = (size_t)lanes * chunks;
  a.part_out = work;
  a.part_peak = work + slots * head_count * head_size;
  a.part_total = a.part_peak + slots * head_count;
  a.q_gain = a.turn = a.k_raw = a.v_raw = a.k_gain = nullptr;
  a.k_ring = a.v_ring = nullptr;
  a.k_code_scale = a.v_code_scale = a.eps = 0.0f;
  dim3 grid(chunks, kv_count, lanes);
  const bool qvec = (((uintptr_t)query) & 15u) == 0 && (q_stride & 3) == 0;
  const TilePlan plan = attend_tile_plan(place0, window, lanes, head_count, head_size);
  if (plan.rb) {
    a.final_out = blend_out;
    a.key_scale = (float)((double)key_scale * unit * score_scale * 1.4426950408889634);  // log2 e
    a.part_peak = work + (size_t)lanes * plan.segments * head_count * head_size;
    a.part_total = a.part_peak + (size_t)lanes * plan.segments * head_count;
    hipError_t e = hipErrorInvalidValue;
    if (head_size == 256 && fmt == 0)
      e = attend_launch_tile<256, 0>(a, plan, kv_count, qvec, stream);
    else if (head_size == 256 && fmt == 1)
      e = attend_launch_tile<256, 1>(a, plan, kv_count, qvec, stream);
    else if (head_size == 512 && fmt == 0)
      e = attend_launch_tile<512, 0>(a, plan, kv_count, qvec, stream);
    else if (head_size == 512 && fmt == 1)
      e = attend_launch_tile<512, 1>(a, plan, kv_count, qvec, stream);
    if (e != hipSuccess || plan.segments == 1) return e;
    return attend_fold(a, plan.segments, 0, place0, place_dev, window, lanes, head_size, blend_out, stream);
  }
  if (head_size == 256 && fmt == 0)
    attend_launch_chunk<256, 0>(a, grid, chunk, qvec, stream);
  else if (head_size == 256 && fmt == 1)
    attend_launch_chunk<256, 1>(a, grid, chunk, qvec, stream);
  else if (head_size == 512 && fmt == 0)
    attend_launch_chunk<512, 0>(a, grid, chunk, qvec, stream);
  else if (head_size == 512 && fmt == 1)
    attend_launch_chunk<512, 1>(a, grid, chunk, qvec, stream);
  else
    return hipErrorInvalidValue;
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || chunks == 1) return e;
  return attend_fold(a, chunks, chunk, place0, place_dev, window, lanes, head_size, blend_out,
                     stream);
}

// The fold of a launch's chunk partials into `blend_out`.
static hipError_t attend_fold(const AttendArgs &a, int chunks, int chunk, int place0,
                              const int *place_dev, int window, int lanes, int head_size,
                              float *blend_out, hipStream_t stream, int extra) {
  const int head_count = a.head_count;
  const int q_stride = a.q_stride;
  // One lane: 16 dims a fold workgroup (the most workgroups); many lanes
  // (a prime or a block): 64.  Chunks a thread loads: enough for one pass.
  const int dims = lanes <= kAttendPrepLanes ? 16 : 64;
  const int slices = 256 / dims;
  int per = 1;
  while (per < 32 && per * slices < chunks) per *= 2;
  const dim3 fgrid(head_count, lanes, head_size / dims);
#define IGL_FOLD(D, P, T)                                                                          \
  hipLaunchKernelGGL((attend_fold_kernel<D, P, T>), fgrid, dim3(256), 0, stream, a.part_out,      \
                     a.part_peak, a.part_total, chunks, chunk, place0, place_dev, window, extra,   \
                     head_count, head_size, blend_out, q_stride)
#define IGL_FOLD_PER(D, T)                                                                         \
  switch (per) {                                                                                   \
    case 1: IGL_FOLD(D, 1, T); break;                                                              \
    case 2: IGL_FOLD(D, 2, T); break;                                                              \
    case 4: IGL_FOLD(D, 4, T); break;                                                              \
    case 8: IGL_FOLD(D, 8, T); break;                                                              \
    case 16: IGL_FOLD(D, 16, T); break;                                                            \
    default: IGL_FOLD(D, 32, T); break;                                                            \
  }
  const bool two = chunk == 0;  // a tile's segments
  if (dims == 16 && two) {
    IGL_FOLD_PER(16, true)
  } else if (dims == 16) {
    IGL_FOLD_PER(16, false)
  } else if (two) {
    IGL_FOLD_PER(64, true)
  } else {
    IGL_FOLD_PER(64, false)
  }
#undef IGL_FOLD_PER
#undef IGL_FOLD
  return hipGetLastError();
}

// The attention of a decode step or a small block with the heads prepared in
// the same launch (attend_split_kernel's PREP form): 1 to kAttendPrepLanes
// lanes, lane 0 at the position in *place_dev (place_bound its upper bound,
// which sizes the grid), e4m3 rings, one key/value head.  query: the query
// heads before their norm, 16-byte aligned, lanes q_stride floats apart (a
// multiple of 4; the blend out the same); turn: lane by lane, turn_stride
// floats apart (a multiple of 4), the (cos, sin) pairs of the lane's position
// times each step, head_size / 2 of them; k_raw, v_raw, k_gain: the key and
// value heads before their norms, lanes kv_stride floats apart, and the key
// gain, whose bytes go to ring slot position % cache_span (NULL for a layer
// that reads another layer's rings and writes none).
extern "C" hipError_t igl_launch_attend_prep(const uint8_t *key_store, const uint8_t *value_store,
                                             float key_scale, float value_scale, int cache_span,
                                             int head_size, int lanes, const float *query,
                                             int q_stride, const float *q_gain, const float *turn,
                                             int turn_stride, const float *k_raw,
                                             const float *v_raw, int kv_stride, const float *k_gain,
                                             uint8_t *k_ring, uint8_t *v_ring, float eps,
                                             int place_bound, const int *place_dev, int window,
                                             float score_scale, float *blend_out, float *work,
                                             hipStream_t stream) {
  AttendArgs a;
  if (lanes < 1 || lanes > kAttendPrepLanes) return hipErrorInvalidValue;
  const int chunk = attend_chunk(place_bound, window, lanes);
  // with k_raw, one slot more a lane: the partial of the block's new positions
  const int extra = k_raw ? 1 : 0;
  const int chunks = attend_blocks(place_bound, window, lanes) + extra;
  if ((((uintptr_t)query) & 15u) || (((uintptr_t)q_gain) & 15u) || (((uintptr_t)turn) & 15u) ||
      !place_dev || !turn)
    return hipErrorInvalidValue;
  if (lanes > 1 && (q_stride < kAttendGroup * head_size || (q_stride & 3) || turn_stride < head_size ||
                    (turn_stride & 3) || (k_raw && kv_stride < head_size)))
    return hipErrorInvalidValue;
  if (k_raw && (!v_raw || !k_gain || !k_ring || !v_ring)) return hipErrorInvalidValue;
  // the new positions of the block sit inside every lane's window and the
  // ring holds them beside every older position a lane reads
  if (window > 0 && lanes > window) return hipErrorInvalidValue;
  if (k_raw && cache_span < (window > 0 ? window : place_bound + 1) + lanes - 1 &&
      cache_span < place_bound + lanes)
    return hipErrorInvalidValue;
  a.key_store = key_store;
  a.value_store = value_store;
  a.kv_width = head_size;
  a.cache_span = cache_span;
  a.place0 = place_bound;
  a.place_dev = place_dev;
  a.window = window;
  a.lanes = lanes;
  a.chunks = chunks;
  a.final_out = chunks == 1 && !extra ? blend_out : nullptr;
  a.q_stride = lanes > 1 ? q_stride : kAttendGroup * head_size;
  a.query = query;
  a.key_scale = key_scale * 256.0f * score_scale;
  a.value_scale = value_scale * 256.0f;
  a.head_count = kAttendGroup;
  a.part_out = work;
  a.part_peak = work + (size_t)lanes * chunks * kAttendGroup * head_size;
  a.part_total = a.part_peak + (size_t)lanes * chunks * kAttendGroup;
  a.q_gain = q_gain;
  a.turn = turn;
  a.turn_stride = lanes > 1 ? turn_stride : 0;
  a.k_raw = k_raw;
  a.kv_raw_stride = lanes > 1 ? kv_stride : 0;
  a.v_raw = v_raw;
  a.k_gain = k_gain;
  a.k_ring = k_ring;
  a.v_ring = v_ring;
  a.k_code_scale = key_scale;
  a.v_code_scale = value_scale;
  a.eps = eps;
  const dim3 grid(chunks, 1, lanes);
  if (head_size == 256 && chunk == 32)
    hipLaunchKernelGGL((attend_split_kernel<256, 0, 32, true, true>), grid, dim3(256), 0, stream, a);
  else if (head_size == 256)
    hipLaunchKernelGGL((attend_split_kernel<256, 0, 64, true, true>), grid, dim3(256), 0, stream, a);
  else if (head_size == 512 && chunk == 32)
    hipLaunchKernelGGL((attend_split_kernel<512, 0, 32, true, true>), grid, dim3(256), 0, stream, a);
  else if (head_size == 512)
    hipLaunchKernelGGL((attend_split_kernel<512, 0, 64, true, true>), grid, dim3(256), 0, stream, a);
  else
    return hipErrorInvalidValue;
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.final_out) return e;
  return attend_fold(a, chunks, chunk, place_bound, place_dev, window, lanes, head_size, blend_out, stream,
                     extra);
}

// Floats of workspace igl_launch_attend_prep needs for the same arguments
// (with key/value rows to write: one partial slot a lane more than the chunks).
extern "C" size_t igl_attend_prep_work_floats(int place_bound, int window, int head_size, int lanes,
                                              int writes_row) {
  const size_t blocks = (size_t)attend_blocks(place_bound, window, lanes) + (writes_row ? 1 : 0);
  return (size_t)lanes * blocks * (size_t)kAttendGroup * ((size_t)head_size + 2);
}

extern "C" int igl_attend_wide(int place0, int window, int lanes) {
  return lanes >= kAttendWideLanes && attend_blocks(place0, window, lanes) > 1;
}

// Floats of workspace igl_launch_attend needs for the same arguments.
extern "C" size_t igl_attend_work_floats(int place0, int window, int lanes, int head_count,
                                         int head_size) {
  const size_t blocks = (size_t)attend_blocks(place0, window, lanes);
  // the tiles' segments, or no partials (below kAttendWideLanes the tiles'
  // segments take no more than the chunks)
  if (igl_attend_wide(place0, window, lanes)) {
    const int segments = attend_tile_plan(place0, window, lanes, head_count, head_size).segments;
    return segments == 1 ? 0 : (size_t)lanes * segments * (size_t)head_count * ((size_t)head_size + 2);
  }
  return (size_t)lanes * blocks * (size_t)head_count * ((size_t)head_size + 2);
}

// Floats of workspace enough for every igl_launch_attend call of at most
// `lanes` lanes whose spans stay within `span_limit` positions.  The chunk
// count is not monotonic in the span: chunks are 32 positions up to
// kAttendShortSpan and 64 beyond, so a span just under kAttendShortSpan has
// more chunks than one just over it.  The largest count of each regime is
// taken.  A launch of kAttendWideLanes lanes and more keeps fewer partials than
// kAttendWideLanes - 1 lanes over the same span (attend_tile_plan).
extern "C" size_t igl_attend_work_floats_limit(int span_limit, int lanes, int head_count,
                                               int head_size) {
  if (span_limit < 1 || lanes < 1) return 0;
  const int short_top = span_limit < kAttendShortSpan ? span_limit : kAttendShortSpan;
  const int b_short = attend_blocks(short_top - 1, 0, 1);
  const int b_long = attend_blocks(span_limit - 1, 0, 1);
  const size_t blocks = (size_t)(b_short > b_long ? b_short : b_long);
  const size_t narrow = (size_t)(lanes < kAttendWideLanes ? lanes : kAttendWideLanes - 1);
  // a prepared launch of up to kAttendPrepLanes lanes (a decode step, a small
  // block) needs blocks + 1 slots a lane: its new positions' partial
  const size_t prep = (size_t)(lanes < kAttendPrepLanes ? lanes : kAttendPrepLanes) * (blocks + 1);
  const size_t slots = narrow * blocks > prep ? narrow * blocks : prep;
  return slots * (size_t)head_count * ((size_t)head_size + 2);
}

// ---- the workspace of the entry that allocates nothing ---------------------
//
// igl_attend_lanes_fixed_dev writes its chunk partials here instead of into
// the desk's grow-only workspace.  One copy of the array lives on each GPU the
// library runs on, until the process ends.  On the host, `scratch` names a
// stand-in, not device memory: host code passes the address that
// hipGetSymbolAddress gives for the current device, resolved once per device
// (igl_attend_fixed_resolve, called by igl_back_open with that device current).
static __device__ __align__(256) float scratch[IGL_ATTEND_FIXED_FLOATS];

namespace {
constexpr int kFixedDevices = 64;
std::mutex fixed_lock;
float *fixed_ptr[kFixedDevices];
}  // namespace

extern "C" hipError_t igl_attend_fixed_resolve(int device) {
  if (device < 0 || device >= kFixedDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> hold(fixed_lock);
  if (fixed_ptr[device]) return hipSuccess;
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  fixed_ptr[device] = static_cast<float *>(ptr);
  return hipSuccess;
}

extern "C" float *igl_attend_fixed_ptr(int device) {
  if (device < 0 || device >= kFixedDevices) return nullptr;
  std::lock_guard<std::mutex> hold(fixed_lock);
  return fixed_ptr[device];
}
