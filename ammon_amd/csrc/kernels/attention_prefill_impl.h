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
// / 8 kv heads of 128, bf16 cache: 2048 tokens 858 -> 101 us (340 TFLOP/s of
// products once each), 301 tokens after 7001 667 -> 104 us; fp32 cache: 1000
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
  uint32_t t0, t1;          // this split's positions, up to the tile's last
  uint32_t row;             // this lane's query row
  uint32_t qpos;            // its position
  uint32_t wmin, wmax;      // positions of the wave's first and last row
  uint32_t head, krow;      // dims, bytes of a cache row
  bool live;                // the wave has rows
  __amdgpu_buffer_rsrc_t kres, vres;

  // Request chunk c into buffer b: each wave four 1 KiB requests of K, four of
  // V.  Rows at or past t1 read as zero.
  AMMON_DEV void stage(char *lds, uint32_t c, uint32_t b) const {
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

  // The eight weights of 16 positions as bf16 parts that sum to them.
  AMMON_DEV static void parts(const f32x16 &p, int kk, bf16x8 (&pp)[3]) {
    const f32x8 f = kk ? __builtin_shufflevector(p, p, 8, 9, 10, 11, 12, 13, 14, 15)
                       : __builtin_shufflevector(p, p, 0, 1, 2, 3, 4, 5, 6, 7);
    pp[0] = __builtin_convertvector(f, bf16x8);
    const f32x8 r1 = f - __builtin_convertvector(pp[0], f32x8);
    pp[1] = __builtin_convertvector(r1, bf16x8);
    pp[2] = __builtin_convertvector(r1 - __builtin_convertvector(pp[1], f32x8), bf16x8);
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
      for (int db = 0; db < DB; ++db) {
        f32x16 t;
#pragma unroll
        for (int i = 0; i < 16; ++i) t[i] = 0.f;
        i16x8 a[2 * SB];
#pragma unroll
        for (int kk = 0; kk < 2 * SB; ++kk) a[kk] = v_frag(vb, kk, db);
#pragma unroll
        for (int q = 2; q >= 0; --q)
#pragma unroll
          for (int kk = 0; kk < 2 * SB; ++kk)
            t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[kk]), pp[kk][q],
                                                        t, 0, 0, 0);
        o[db] += t;
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

  // A masked weight is 0, and 0 times an infinity or NaN is not: where a chunk
  // holds positions past some row's own, V of a later token must not reach the
  // earlier one.  True if the chunk's V has such an element.
  AMMON_DEV bool values_not_finite(const char *vb) const {
    uint32_t bad = 0;
#pragma unroll 2
    for (uint32_t i = lane; i < HALF / 16; i += 64) {
      const u32x4 v = ((const u32x4 *)vb)[i];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        bad |= BF ? ((v[e] & 0x7f807f80u) + 0x00800080u) & 0x80008000u
                  : ((v[e] & 0x7f800000u) + 0x00800000u) & 0x80000000u;
    }
    return __any(bad != 0);
  }

  // ... and then the wave's rows are computed one by one from the cache, up to
  // each row's own position (lane: dims 2 lane and 2 lane + 1).
  AMMON_DEV void rows_one_by_one(const ammon_k_attention &p, uint32_t g, uint32_t split,
                                 uint32_t w0) const {
    const uint32_t G = p.q_heads / p.kv_heads, rows = p.tokens * G, d = 2 * lane;
    const float scale2 = 1.4426950408889634f / sqrtf((float)head);
#pragma unroll 1
    for (uint32_t r = w0; r < min(w0 + 32, rows); ++r) {
      const uint32_t token = r / G, qh = g * G + (r - token * G);
      const uint32_t pos = p.step->position + token;
      const size_t at = (size_t)token * p.q_heads + qh;
      const bool mine = d < head, ok = pos < p.limit;
      float q0 = 0.f, q1 = 0.f, m = -INFINITY, l = 0.f, o0 = 0.f, o1 = 0.f;
      if (mine) q0 = p.q[at * head + d], q1 = p.q[at * head + d + 1];
#pragma unroll 1
      for (uint32_t t = t0; ok && t < t1 && t <= pos; ++t) {
        const size_t k = ((size_t)g * p.seq + t) * head + (mine ? d : 0);
        const float k0 = load_elem(p.k_cache, DTYPE, k), k1 = load_elem(p.k_cache, DTYPE, k + 1);
        const float v0 = load_elem(p.v_cache, DTYPE, k), v1 = load_elem(p.v_cache, DTYPE, k + 1);
        const float s = wave_sum(mine ? q0 * k0 + q1 * k1 : 0.f) * scale2;
        const float mn = fmaxf(m, s), mu = mn == -INFINITY ? 0.f : mn;
        const float a = __builtin_amdgcn_exp2f(m - mu), e = __builtin_amdgcn_exp2f(s - mu);
        l = l * a + e;
        o0 = o0 * a + e * v0;
        o1 = o1 * a + e * v1;
        m = mn;
      }
      if (p.splits == 1) {
        const float nan = __uint_as_float(0x7fc00000u);
        if (mine)
          *(float2 *)(p.out + at * head + d) = ok ? make_float2(o0 / l, o1 / l) : make_float2(nan, nan);
      } else if (ok && t0 <= pos) {
        float *w = p.partial + (at * p.splits + split) * (head + 2);
        if (mine) *(float2 *)(w + d) = make_float2(o0, o1);
        if (lane == 0) *(float2 *)(w + head) = make_float2(m * 0.6931471805599453f, l);
      }
    }
  }

  // Rows [128 tile, +128) of kv head g over split `split`.
  AMMON_DEV void run(const ammon_k_attention &p, uint32_t g, uint32_t tile, uint32_t split,
                     char *lds) {
    lane = threadIdx.x & 63;
    h = lane >> 5;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    head = p.head;
    krow = head * (uint32_t)sizeof(KV);
    const uint32_t start = p.step->position;
    const uint32_t G = p.q_heads / p.kv_heads, rows = p.tokens * G;
    const uint32_t w0 = tile * PF_ROWS + 32 * wave;  // the wave's first row
    live = w0 < rows;
    wmin = start + (live ? w0 : rows - 1) / G;
    wmax = start + min(w0 + 31, rows - 1) / G;
    row = w0 + (lane & 31);
    const uint32_t token = min(row, rows - 1) / G;
    const uint32_t qh = g * G + (min(row, rows - 1) - token * G);
    qpos = start + token;
    const uint32_t last = start + min(tile * PF_ROWS + PF_ROWS - 1, rows - 1) / G;
    t0 = split * p.split_len;
    t1 = min(min(last + 1, t0 + p.split_len), p.limit);
    const bool direct = p.splits == 1;
    float *out = p.out + ((size_t)token * p.q_heads + qh) * head;
    if (t0 >= t1) {  // no position of this range is live for any row (uniform)
      return;
    }
    kres = make_rsrc((const KV *)p.k_cache + ((size_t)g * p.seq + t0) * head, (t1 - t0) * krow);
    vres = make_rsrc((const KV *)p.v_cache + ((size_t)g * p.seq + t0) * head, (t1 - t0) * krow);

    // q: B operand, lane = row; fragment kk holds dims 16 kk + 8 h..+7 (fp32:
    // 8 kk + 4 h..+3); dims past the head are zero
    const float *qp = p.q + ((size_t)token * p.q_heads + qh) * head;
    bf16x8 qb[BF ? QF : 1][NQ];
    f32x4 qf[BF ? 1 : QF];
    if constexpr (BF) {
#pragma unroll
      for (int kk = 0; kk < QF; ++kk) {
        const uint32_t d = 16 * kk + 8 * h;
        f32x8 f = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (d < head) {
          const float4 a = ld_in4(qp + d), b = ld_in4(qp + d + 4);
          f = f32x8{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        }
#pragma unroll
        for (int part = 0; part < NQ; ++part) {
          qb[kk][part] = __builtin_convertvector(f, bf16x8);
          f = f - __builtin_convertvector(qb[kk][part], f32x8);
        }
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < QF; ++kk) {
        const uint32_t d = 8 * kk + 4 * h;
        qf[kk] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (d < head) {
          const float4 a = ld_in4(qp + d);
          qf[kk] = f32x4{a.x, a.y, a.z, a.w};
        }
      }
    }
    stage(lds, 0, 0);

    const float scale2 = 1.4426950408889634f / sqrtf((float)head);  // log2(e) / sqrt(head)
    f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
    float m = -INFINITY, l = 0.f;  // l: this lane's positions only, summed at the end
    const uint32_t lim = min(qpos, t1 - 1);  // last position of this lane's row
    const uint32_t kat = (lane & 31) * ROW + ((h ^ (lane & (SLOTS - 1) & 31)) << 4);

    bool tainted = false;
    const uint32_t nch = (t1 - t0 + CH - 1) / CH;
    for (uint32_t c = 0; c < nch; ++c) {
      wait_vmcnt<0>();
      __syncthreads();  // chunk c has landed; the other buffer is consumed
      if (c + 1 < nch) stage(lds, c + 1, (c + 1) & 1);
      const uint32_t first = t0 + c * CH;
      if (!live || first > wmax) continue;  // uniform per wave
      const char *kb = lds + (c & 1) * 2 * HALF, *vb = kb + HALF;
      f32x16 s[SB], sp[2];  // sp: sums of their own (short chains of fp32 additions)
#pragma unroll
      for (int b = 0; b < SB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[b][i] = sp[b][i] = 0.f;
#pragma unroll
      for (int kk = 0; kk < QF; ++kk) {
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
      if (__any(mc > m + PF_SLACK)) {
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
      if (masked && values_not_finite(vb)) tainted = true;
      values(vb, s, o);
    }
    if (tainted) {  // uniform per wave
      rows_one_by_one(p, g, split, w0);
      return;
    }
    l = pair32_sum(l);
    if (!live || row >= rows) return;
    if (direct) {
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
    float *w = p.partial + ((size_t)token * p.q_heads * p.splits + (size_t)qh * p.splits + split) * (head + 2);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const uint32_t d = 32 * db + 8 * (i >> 2) + 4 * h + (i & 3);
        if (d < head) *(float2 *)(w + d) = make_float2(o[db][i], o[db][i + 1]);
      }
    if (h == 0) *(float2 *)(w + head) = make_float2(m * 0.6931471805599453f, l);  // natural-log units
  }
};
