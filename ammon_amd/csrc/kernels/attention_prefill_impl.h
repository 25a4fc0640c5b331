// attention_prefill_impl.h -- attention of many consecutive query tokens
// (prompt prefill) on matrix cores, K and V read once per tile of query rows.
//
// Reference semantics as attention_impl.h's (src/kernels.rs:228-410): row
// (token, q head) attends to positions 0..step->position + token of its kv
// head.  The query rows of one kv head are numbered token * G + head in
// group, so a G:1 group's heads share every K and V byte as in decode, and
// so do neighbouring tokens.
//
// A workgroup owns PF_ROWS = 128 of these rows, 32 per wave, over one range of
// positions (split), and walks it in chunks of 64 (bf16) or 32 (fp32)
// positions.  K and V of a chunk are requested straight into LDS, one chunk
// ahead (two buffers of 32 KiB, one barrier per chunk), and read by all four
// waves.  Per chunk a wave computes, on 32x32 tiles:
//   scores  S^T[t][row] = K[t] . q[row]: A = K rows from LDS, B = the wave's q,
//           held in registers.  bf16 K: q as bf16 hi + lo (~16 bits, fp32
//           accumulation) as in decode; fp32 K: fp32 products.
//   weights P = 2^(s log2e / sqrt(head) - m), exact fp32 values; the reference
//           maximum m of a row moves only when a chunk exceeds it by more than
//           PF_SLACK (P then stays below 2^PF_SLACK: no precision is lost, and
//           the output tiles are rarely rescaled);
//   values  O^T[d][row] += V[t][d] P[row][t]: the score tile's registers are the
//           B operand as they stand (its k order, 4 (l / 32) + i then + 8, is
//           taken by the V reads too); bf16 V: A by transposing LDS reads, P
//           as three bf16 parts that sum to it exactly; fp32 V: fp32 products.
// With one split a workgroup writes the result, otherwise the partial of its
// range, which ammon_attention_combine_waves merges.
//
// fp32 sums are kept in short chains: 16, 32 or 64 positions' products by
// themselves, then one addition per output, over splits of at most 2048
// positions.  So the error against 64 bits is no larger than that of one unit
// per token (decode's), also at long contexts: 8:1 heads of 128, bf16 cache,
// 32768 positions, root mean square of the result: 2.52e-6 (unit 2.53e-6; every
// product of a split of any length in one sum: 3.10e-6); 6:1: 2.43e-7 (2.57e-7;
// 6.38e-7); fp32 cache, 8:1: 2.45e-7 (2.92e-7; 6.45e-7).
//
// What bounds it.  Matrix work: per (row, position) pair 2 of the score
// products and 3 of the value products, 2.5 times the bf16 minimum, and about
// as many VALU cycles for the weights and their parts, which the second
// workgroup of a CU overlaps.  One unit per (token, kv head) fills 4 of 16
// columns of each tile at 4:1 and reads K and V once per token.  Measured, 32 q
// / 8 kv heads of 128, bf16 cache: 2048 tokens 858 -> 97 us (354 TFLOP/s of
// products once each), 301 tokens after 7001 667 -> 105 us; fp32 cache: 1000
// tokens 352 -> 153 us.
//
// Rows land in LDS with their 16-byte pieces XOR-swizzled: K piece p of row r
// at slot p ^ r (the score operand reads one piece of 32 rows), bf16 V at
// p ^ 4 (r % 4) (a half wave's transposing read takes four rows' 64 bytes),
// fp32 V at p ^ 8 (r / 4 % 2) (a read takes 128 bytes of rows r and r + 4).  A
// head below 128 keeps the row stride; pieces past it read as zero.
#pragma once

#include "attention_impl.h"

#define PF_ROWS 128
#define PF_SLACK 8.0f

// DB: ceil(head / 32); NQ: bf16 parts of q (bf16 K/V)
template <typename KV, int DB, int NQ>
struct PrefillTile {
  typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
  typedef short i16x4 __attribute__((ext_vector_type(4)));
  typedef short i16x8 __attribute__((ext_vector_type(8)));
  typedef float f32x8 __attribute__((ext_vector_type(8)));
  typedef float f32x16 __attribute__((ext_vector_type(16)));

  static constexpr bool BF = sizeof(KV) == 2;
  static constexpr uint32_t DTYPE = BF ? AMMON_K_BF16 : AMMON_K_F32;
  static constexpr uint32_t CH = BF ? 64 : 32;       // positions per chunk
  static constexpr int SB = CH / 32;                 // 32-position score tiles
  static constexpr uint32_t SLOTS = BF ? 16 : 32;    // 16-byte slots per LDS row
  static constexpr uint32_t ROW = SLOTS * 16;        // bytes
  static constexpr uint32_t HALF = CH * ROW;         // K (or V) of a chunk: 16 KiB
  static constexpr int QF = BF ? 2 * DB : 4 * DB;    // q fragments: 16 (8) dims each

  uint32_t lane, h, wave;
  uint32_t g;               // kv head
  uint32_t t0, t1;          // this split's positions, up to the tile's last
  uint32_t row;             // this lane's query row
  uint32_t qpos;            // its position
  uint32_t wmin, wmax;      // positions of the wave's first and last row
  uint32_t head, krow;      // dims, bytes of a cache row
  bool live;                // the wave has rows
  __amdgpu_buffer_rsrc_t kres, vres;
  bf16x8 qb[BF ? QF : 1][NQ];  // q, the score products' B operand
  f32x4 qf[BF ? 1 : QF];

  // This lane's row in q and out ([tokens, q heads]; past the last: the last).
  AMMON_DEV size_t row_at(const ammon_k_attention &p) const {
    const uint32_t G = p.q_heads / p.kv_heads, r = min(row, p.tokens * G - 1), token = r / G;
    return (size_t)token * p.q_heads + g * G + (r - token * G);
  }

  // q fragment kk of a row: dims 16 kk + 8 h..+7 in NQ bf16 parts (fp32:
  // 8 kk + 4 h..+3); dims past the head are zero.
  AMMON_DEV void q_frag(const float *q, int kk, bf16x8 (&part)[NQ]) const {
    const uint32_t d = 16 * kk + 8 * h, at = min(d, head - 8);
    const float4 a = ld_in4(q + at), b = ld_in4(q + at + 4);
    f32x8 f = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    if (d >= head) f = f32x8{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      part[i] = __builtin_convertvector(f, bf16x8);
      f = f - __builtin_convertvector(part[i], f32x8);
    }
  }
  AMMON_DEV f32x4 q_frag(const float *q, int kk) const {
    const uint32_t d = 8 * kk + 4 * h;
    const float4 a = ld_in4(q + min(d, head - 4));
    return d < head ? f32x4{a.x, a.y, a.z, a.w} : f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // Request chunk c into buffer b: each wave four 1 KiB requests of K, four of
  // V.  Rows at or past t1 read as zero.
  AMMON_DEV void stage(char *lds, uint32_t c, uint32_t b, uint32_t lane) const {
    const uint32_t s = lane & (SLOTS - 1);
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t r = (wave * 4 + i) * (64 / SLOTS) + lane / SLOTS;
        const uint32_t t = c * CH + r;
        const uint32_t piece = v == 0 ? s ^ (r & (SLOTS - 1)) : BF ? s ^ (4 * (r & 3)) : s ^ (8 * (r >> 2 & 1));
        const uint32_t off = t < t1 - t0 && piece * 16 < krow ? t * krow + piece * 16 : AMMON_OOB;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            v == 0 ? kres : vres,
            (__attribute__((address_space(3))) void *)(lds + b * 2 * HALF + v * HALF + (wave * 4 + i) * 1024),
            16, off, 0, 0, 0);
      }
  }

  // A operand kk of the value product of dims 32 db..+31 (bf16: 16 positions
  // 16 kk.. in the order 4h + i, 8 + 4h + i; lane = dim).
  AMMON_DEV i16x8 v_frag(const char *vb, int kk, int db) const {
    const uint32_t s = lane & 15;
    const uint32_t slot = (4 * (s >> 2)) | (2 * (lane >> 4 & 1)) | ((s >> 1) & 1);
    const uint32_t at = ((4 * h + (s >> 2)) * ROW + slot * 16 + (s & 1) * 8) ^ (db << 6);
    typedef __attribute__((address_space(3))) i16x4 *tr;
    const i16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr)(vb + at + kk * 16 * ROW));
    const i16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr)(vb + at + (kk * 16 + 8) * ROW));
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
  }
  // fp32: lane = dim, position 8 (i / 4) + 4h + i % 4.
  AMMON_DEV float v_elem(const char *vb, int i, int db) const {
    const uint32_t l = lane & 31;
    const uint32_t at = (4 * h * ROW + (((l >> 2) ^ (8 * h)) * 16) + (l & 3) * 4) ^ (db << 7);
    return *(const float *)(vb + at + (8 * (i >> 2) + (i & 3)) * ROW);
  }

  // Two floats as bf16, and what they leave.  (Pair by pair: from eight at a time
  // the compiler rounded every element a second time to widen it, 64 instructions
  // a chunk.)
  AMMON_DEV static uint32_t part2(float &a, float &b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
    a -= bf16_lo(w);
    b -= bf16_hi(w);
    return w;
  }

  // The eight weights of 16 positions as bf16 parts that sum to them.
  AMMON_DEV static void parts(const f32x16 &p, int kk, bf16x8 (&pp)[3]) {
    u32x4 w[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float a = p[8 * kk + 2 * e], b = p[8 * kk + 2 * e + 1];
#pragma unroll
      for (int q = 0; q < 3; ++q) w[q][e] = part2(a, b);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) pp[q] = __builtin_bit_cast(bf16x8, w[q]);
  }

  // O += V P of one chunk.  32 or 64 positions' products are summed by
  // themselves, small parts first, and then added to the output once: a sum that
  // takes every product rounds 12 times per chunk at the output's size.  The
  // matrix unit's bf16 sums round downwards (measured: 32768 positions of
  // zero-mean V gave outputs 2e-7 of their size too low), so with q whole, where
  // that shows, every second sum is taken of -P and subtracted.
  AMMON_DEV void values(const char *vb, const f32x16 (&p)[SB], f32x16 (&o)[DB]) const {
    if constexpr (BF && NQ == 2) {
      bf16x8 pp[2 * SB][3];
#pragma unroll
      for (int kk = 0; kk < 2 * SB; ++kk) parts(p[kk / 2], kk & 1, pp[kk]);
#pragma unroll
      for (int db = 0; db < DB; db += 2) {
        // two chains in turn (one block of dims at a time: 2048 tokens 97 -> 99 us)
        f32x16 t[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) t[0][i] = t[1][i] = 0.f;
#pragma unroll
        for (int kk = 0; kk < 2 * SB; ++kk) {
          const i16x8 a[2] = {v_frag(vb, kk, db), v_frag(vb, kk, db + 1)};
#pragma unroll
          for (int q = 2; q >= 0; --q)
#pragma unroll
            for (int e = 0; e < 2; ++e)
              t[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[e]),
                                                             pp[kk][q], t[e], 0, 0, 0);
        }
        o[db] += t[0];
        o[db + 1] += t[1];
        __builtin_amdgcn_sched_barrier(0);  // no reading ahead: registers
      }
    } else if constexpr (BF) {
#pragma unroll
      for (int b = 0; b < SB; ++b) {
        bf16x8 pp[2][3];
        const f32x16 pb = b & 1 ? -p[b] : p[b];
        parts(pb, 0, pp[0]);
        parts(pb, 1, pp[1]);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          f32x16 t;
#pragma unroll
          for (int i = 0; i < 16; ++i) t[i] = 0.f;
          const i16x8 a[2] = {v_frag(vb, 2 * b, db), v_frag(vb, 2 * b + 1, db)};
#pragma unroll
          for (int q = 2; q >= 0; --q)
#pragma unroll
            for (int k = 0; k < 2; ++k)
              t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[k]), pp[k][q],
                                                          t, 0, 0, 0);
          if (b & 1)
            o[db] -= t;
          else
            o[db] += t;
        }
        __builtin_amdgcn_sched_barrier(0);  // no reading ahead: registers
      }
    } else {
      // the sums of 16 positions each, then one addition per output (short
      // chains)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        f32x16 t[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) t[0][i] = t[1][i] = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i)
          t[i / 8] = __builtin_amdgcn_mfma_f32_32x32x2f32(v_elem(vb, i, db), p[0][i], t[i / 8], 0, 0, 0);
        o[db] += t[0] + t[1];
        __builtin_amdgcn_sched_barrier(0);  // one tile's V reads in flight: registers
      }
    }
  }

  // ---- elements that are not finite ----------------------------------------
  // The products of a chunk are right for finite K and V only: the parts of q and P
  // have signs of their own (inf x mid may be -inf), and a masked weight is 0,
  // which an infinity turns into NaN, so that V of a later token would reach an
  // earlier one.  Any of it leaves a result that is not finite, so the wave looks
  // at its results once, at the end, and repeats the split (again() in run) where
  // one is not.  The second walk keeps weights at or below 1, as the units do,
  // multiplies zeros in place of such elements and counts them apart: per result, count 1024 for every such element and its sign for
  // every infinity (x sign of q, x 1 for a weight above 0).  Counts are whole
  // numbers below 2^24: exact.
  struct Split {
    u32x4 finite, count, sign;  // bf16 pairs
  };
  AMMON_DEV static Split split(u32x4 v) {
    Split s;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t w = v[e];
      const uint32_t bad = ((w & 0x7f807f80u) + 0x00800080u) & 0x80008000u;
      const uint32_t nan = (((w & 0x007f007fu) + 0x007f007fu) & 0x00800080u) << 8 & bad;
      const uint32_t all = (bad >> 15) * 0xffffu, inf = ((bad ^ nan) >> 15) * 0xffffu;
      s.finite[e] = w & ~all;
      s.count[e] = all & 0x44804480u;                        // 1024
      s.sign[e] = inf & ((w & 0x80008000u) | 0x3f803f80u);   // +-1
    }
    return s;
  }
  AMMON_DEV static void split(float v, float &finite, float &count, float &sign) {
    const uint32_t u = __float_as_uint(v) & 0x7fffffffu;
    finite = u >= 0x7f800000u ? 0.f : v;
    count = u >= 0x7f800000u ? 1024.f : 0.f;
    sign = u == 0x7f800000u ? copysignf(1.f, v) : 0.f;
  }
  // What those elements add to the result they were counted for.
  AMMON_DEV static float counted(float e) {
    const float n = rintf(e * (1.f / 1024.f)), d = fmaf(-1024.f, n, e);
    float r = __uint_as_float(0x7fc00000u);
    r = d == n ? INFINITY : r;
    r = d == -n ? -INFINITY : r;
    return e == 0.f ? 0.f : r;
  }
  AMMON_DEV static f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.f;
    return z;
  }
  AMMON_DEV static f32x16 mfma_bf16(u32x4 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), b, c, 0, 0, 0);
  }

  // Scores and values of a chunk that may hold such elements (q is read again:
  // registers).
  AMMON_DEV void scores_counted(const ammon_k_attention &p, const char *kb, uint32_t kat,
                                f32x16 (&s)[SB]) const {
    size_t at = row_at(p) * head;
    asm volatile("" : "+v"(at));  // not ahead of the chunk loop: registers
    const float *q = p.q + at;
#pragma unroll
    for (int b = 0; b < SB; ++b) {
      f32x16 hi = zero16(), rest = zero16(), n = zero16();
#pragma unroll
      for (int kk = 0; kk < QF; ++kk) {
        const char *ka = kb + (kat ^ (kk << 5)) + b * 32 * ROW;
        if constexpr (BF) {
          const Split a = split(*(const u32x4 *)ka);
          bf16x8 qk[NQ];
          q_frag(q, kk, qk);
          u32x4 sign = __builtin_bit_cast(u32x4, qk[0]), one;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t w = sign[e], set = ((w & 0x7fff7fffu) + 0x7fff7fffu) & 0x80008000u;
            sign[e] = (set >> 15) * 0xffffu & ((w & 0x80008000u) | 0x3f803f80u);
            one[e] = 0x3f803f80u;
          }
#pragma unroll
          for (int part = 0; part < NQ; ++part) {
            f32x16 &acc = part ? rest : hi;
            acc = mfma_bf16(a.finite, qk[part], acc);
          }
          n = mfma_bf16(a.count, __builtin_bit_cast(bf16x8, one), n);
          n = mfma_bf16(a.sign, __builtin_bit_cast(bf16x8, sign), n);
        } else {
          const f32x4 a = *(const f32x4 *)ka, qk = q_frag(q, kk);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float finite, count, sign;
            split(a[e], finite, count, sign);
            f32x16 &acc = kk & 1 ? rest : hi;
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(finite, qk[e], acc, 0, 0, 0);
            n = __builtin_amdgcn_mfma_f32_32x32x2f32(count, 1.f, n, 0, 0, 0);
            n = __builtin_amdgcn_mfma_f32_32x32x2f32(
                sign, qk[e] == 0.f ? 0.f : copysignf(1.f, qk[e]), n, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);  // (registers, here and below)
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) s[b][i] = hi[i] + rest[i] + counted(n[i]);
    }
  }

  AMMON_DEV void values_counted(const char *vb, const f32x16 (&p)[SB], uint32_t first, uint32_t lim,
                                f32x16 (&o)[DB]) const {
#pragma unroll
    for (int b = 0; b < SB; ++b) {
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        f32x16 t = zero16(), n = zero16();
        if constexpr (BF) {
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const Split a = split(__builtin_bit_cast(u32x4, v_frag(vb, 2 * b + k, db)));
            bf16x8 pp[3];
            parts(p[b], k, pp);
#pragma unroll
            for (int q = 2; q >= 0; --q) t = mfma_bf16(a.finite, pp[q], t);
            u32x4 live, above;  // bf16 ones
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const uint32_t i = 8 * k + 2 * e, at = first + 32 * b + 8 * (i >> 2) + 4 * h + (i & 3);
              live[e] = (at <= lim ? 0x3f80u : 0u) | (at + 1 <= lim ? 0x3f800000u : 0u);
              above[e] = live[e] & ((p[b][i] > 0.f ? 0xffffu : 0u) | (p[b][i + 1] > 0.f ? 0xffff0000u : 0u));
            }
            n = mfma_bf16(a.count, __builtin_bit_cast(bf16x8, live), n);
            n = mfma_bf16(a.sign, __builtin_bit_cast(bf16x8, above), n);
            __builtin_amdgcn_sched_barrier(0);
          }
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            float finite, count, sign;
            split(v_elem(vb, i, db), finite, count, sign);
            const float live = first + 8 * (i >> 2) + 4 * h + (i & 3) <= lim ? 1.f : 0.f;
            t = __builtin_amdgcn_mfma_f32_32x32x2f32(finite, p[b][i], t, 0, 0, 0);
            n = __builtin_amdgcn_mfma_f32_32x32x2f32(count, live, n, 0, 0, 0);
            n = __builtin_amdgcn_mfma_f32_32x32x2f32(sign, p[b][i] > 0.f ? live : 0.f, n, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = o[db][i] + t[i] + counted(n[i]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // The split's chunks for the wave's rows (go: or only its share of the
  // staging): m, l and o of each row.  CARE: the second walk, above.
  template <bool CARE>
  AMMON_DEV void walk(const ammon_k_attention &p, char *lds, bool go, f32x16 (&o)[DB], float &m,
                      float &l) const {
    const float scale2 = 1.4426950408889634f / sqrtf((float)head);  // log2(e) / sqrt(head)
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] = zero16();
    m = -INFINITY, l = 0.f;  // l: this lane's positions only, summed at the end
    const uint32_t lim = min(qpos, t1 - 1);  // last position of this lane's row
    stage(lds, 0, 0, lane);
    const uint32_t nch = (t1 - t0 + CH - 1) / CH;
    for (uint32_t c = 0; c < nch; ++c) {
      wait_vmcnt<0>();
      __syncthreads();  // chunk c has landed; the other buffer is consumed
      uint32_t ln = lane;
      if (CARE || (NQ == 3 && DB == 3))  // offsets computed again, not kept: registers
        asm volatile("" : "+v"(ln));
      if (c + 1 < nch) stage(lds, c + 1, (c + 1) & 1, ln);
      const uint32_t first = t0 + c * CH;
      if (!go || !live || first > wmax) continue;  // uniform per wave
      const char *kb = lds + (c & 1) * 2 * HALF, *vb = kb + HALF;
      f32x16 s[SB], sp[2];  // sp: sums of their own (short chains of fp32 additions)
#pragma unroll
      for (int b = 0; b < SB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[b][i] = sp[b][i] = 0.f;
      const uint32_t kat = (ln & 31) * ROW + (((ln >> 5) ^ (ln & (SLOTS - 1) & 31)) << 4);
      if constexpr (CARE) scores_counted(p, kb, kat, s);
#pragma unroll
      for (int kk = 0; kk < (CARE ? 0 : QF); ++kk) {
        if constexpr (BF) {
          bf16x8 a[SB];
#pragma unroll
          for (int b = 0; b < SB; ++b)
            a[b] = *(const bf16x8 *)(kb + (kat ^ (kk << 5)) + b * 32 * ROW);
#pragma unroll
          for (int part = 0; part < NQ; ++part)
#pragma unroll
            for (int b = 0; b < SB; ++b) {
              f32x16 &acc = NQ == 3 && part ? sp[b] : s[b];
              acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[b], qb[kk][part], acc, 0, 0, 0);
            }
          if (NQ == 3 && kk == QF - 1)
#pragma unroll
            for (int b = 0; b < SB; ++b) s[b] += sp[b];
        } else {  // 16 dims each, summed in pairs
          const f32x4 a = *(const f32x4 *)(kb + (kat ^ (kk << 5)));
          f32x16 &acc = sp[kk / 2 % 2];
          if (kk % 2 == 0)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], qf[kk][e], acc, 0, 0, 0);
          if (kk % 4 == 3) s[0] += sp[0] + sp[1];
        }
      }
      // lane: its row's scores at positions first + 32 b + 8 (i / 4) + 4 h + i % 4
      const bool masked = first + CH - 1 > min(wmin, t1 - 1);  // uniform
      if (masked) {
#pragma unroll
        for (int b = 0; b < SB; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (first + 32 * b + 8 * (i >> 2) + 4 * h + (i & 3) > lim) s[b][i] = -INFINITY;
      }
      float mc = s[0][0];
#pragma unroll
      for (int b = 0; b < SB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) mc = fmaxf(mc, s[b][i]);
      mc = pair32_max(mc) * scale2;
      if (__any(mc > (CARE ? m : m + PF_SLACK))) {
        const float mn = fmaxf(m, mc);
        const float sc = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mn);
#pragma unroll
        for (int db = 0; db < DB; ++db) o[db] *= sc;
        l *= sc;
        m = mn;
      }
      // a row with no position yet keeps (m, l, o) = (-inf, 0, 0)
      const float mu = m == -INFINITY ? 0.f : m;
      float ls[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < SB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[b][i] = __builtin_amdgcn_exp2f(fmaf(s[b][i], scale2, -mu));
          ls[i & 3] += s[b][i];
        }
      l += (ls[0] + ls[1]) + (ls[2] + ls[3]);
      if constexpr (CARE)
        values_counted(vb, s, first, lim, o);
      else
        values(vb, s, o);
    }
  }

  // The result or partial of each row.
  AMMON_DEV void finish(const ammon_k_attention &p, uint32_t split, const f32x16 (&o)[DB], float m,
                        float l) const {
    l = pair32_sum(l);
    if (!live || row >= p.tokens * (p.q_heads / p.kv_heads)) return;
    if (p.splits == 1) {
      float *out = p.out + row_at(p) * head;
      const bool ok = qpos < p.limit;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
          const uint32_t d = 32 * db + 2 * i + 4 * h;
          if (d >= head) continue;
          float4 v;
          v.x = o[db][i] / l, v.y = o[db][i + 1] / l, v.z = o[db][i + 2] / l, v.w = o[db][i + 3] / l;
          const float nan = __uint_as_float(0x7fc00000u);
          if (!ok) v = make_float4(nan, nan, nan, nan);
          *(float4 *)(out + d) = v;
        }
      return;
    }
    if (qpos >= p.limit || t0 > qpos) return;  // dead for this row: the merge skips it
    float *w = p.partial + (row_at(p) * p.splits + split) * (head + 2);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const uint32_t d = 32 * db + 8 * (i >> 2) + 4 * h + (i & 3);
        if (d < head) *(float2 *)(w + d) = make_float2(o[db][i], o[db][i + 1]);
      }
    if (h == 0) *(float2 *)(w + head) = make_float2(m * 0.6931471805599453f, l);  // natural-log units
  }

  // Rows [128 tile, +128) of kv head g over split `split`.
  AMMON_DEV void run(const ammon_k_attention &p, uint32_t g_, uint32_t tile, uint32_t split,
                     char *lds) {
    g = g_;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    head = p.head;
    krow = head * (uint32_t)sizeof(KV);
    const uint32_t start = p.step->position;
    const uint32_t G = p.q_heads / p.kv_heads, rows = p.tokens * G;
    const uint32_t w0 = tile * PF_ROWS + 32 * wave;  // the wave's first row
    live = w0 < rows;
    wmin = start + (live ? w0 : rows - 1) / G;
    wmax = start + min(w0 + 31, rows - 1) / G;
    auto lanes = [&] {
      uint32_t tid = threadIdx.x;
      asm volatile("" : "+v"(tid));  // computed again, not kept across a walk: registers
      lane = tid & 63;
      h = lane >> 5;
      row = w0 + (lane & 31);
      qpos = start + min(row, rows - 1) / G;
    };
    lanes();
    const uint32_t last = start + min(tile * PF_ROWS + PF_ROWS - 1, rows - 1) / G;
    t0 = split * p.split_len;
    t1 = min(min(last + 1, t0 + p.split_len), p.limit);
    if (t0 >= t1) {  // no position of this range is live for any row (uniform)
      return;
    }
    kres = make_rsrc((const KV *)p.k_cache + ((size_t)g * p.seq + t0) * head, (t1 - t0) * krow);
    vres = make_rsrc((const KV *)p.v_cache + ((size_t)g * p.seq + t0) * head, (t1 - t0) * krow);

    const float *q = p.q + row_at(p) * head;
#pragma unroll
    for (int kk = 0; kk < QF; ++kk) {
      if constexpr (BF)
        q_frag(q, kk, qb[kk]);
      else
        qf[kk] = q_frag(q, kk);
    }

    f32x16 o[DB];
    float m, l;
    walk<false>(p, lds, true, o, m, l);
    lanes();
    // again? (what decides it: a row whose result is read)
    float z = l * 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) z = fmaf(o[db][i], 0.f, z);
    const uint64_t off = __ballot(live && row < rows && qpos < p.limit && t0 <= qpos && !(z == 0.f));
    if (!off) finish(p, split, o, m, l);
    __syncthreads();  // the ring is consumed
    if (lane == 0) ((uint32_t *)lds)[wave] = (uint32_t)off | (uint32_t)(off >> 32);
    __syncthreads();
    const u32x4 any = *(const u32x4 *)lds;
    if (!(any[0] | any[1] | any[2] | any[3])) return;  // uniform: every wave stages
    __syncthreads();
    walk<true>(p, lds, off != 0, o, m, l);
    lanes();
    if (off) finish(p, split, o, m, l);
  }
};
