// Decode attention with one sequence's keys over many workgroups, for long
// contexts and small batches, bit-equal to the block walk of
// kernels/attention_gqa.h:404-547 / ref_qwen3.py:210-266.
//
// k_attn_decode.hip gives a sequence one workgroup per head (or per KV head),
// which walks the key blocks chunk by chunk: a 4000-key context is six serial
// chunks of ~6 us on 16 of 256 CUs.  Of the recurrence only the den/res chain
// is sequential, and it is two operations per block and dimension; everything
// else needs a block and the running maximum, a prefix max of the block
// maxima.  So three launches, each over every (sequence, KV head, 4 blocks):
//   score  one wave per block: S = q8.k8^T of the KV head's two query heads,
//          s and the block maxima to the workspace; its prologue is the head
//          epilogue of the new token's projection rows (Q, K: RMSNorm, RoPE,
//          quant; V: quant), the workgroup of the last block writing the page
//          slot
//   pv     one wave per block: nmm_j = max of the block maxima 0..j, P =
//          exp(s - nmm_j), psum_j, P8, pv_j = f32(P8.V) * pmax_j to the
//          workspace
//   chain  one workgroup per (sequence, head): corr_j = exp(nmm_{j-1} -
//          nmm_j), den = den * corr_j + psum_j, res = res * corr_j + pv_j in
//          block order, then the output quantisation
// with the reference's rounding points.  At 4000 keys and b = 1 the launches
// take 4.5, 5.0 and 7.1 us (the fused launch they replace, with its down and
// Q|K|V projections: 43.6), at 24 rows x 2048 keys 14.8, 15.5 and 6.3 us;
// score and pv are bound by latency below ~1000 blocks, then by the K and V
// stream (3.4 TB/s), chain by the walk over the blocks (one per ~30 cycles).
// Two or four blocks per wave were slower at every size (24 x 2048: 1998 us a
// step against 2109 and 2268), and so was prefetching the next GEMVs' weights
// beside pv and chain (4000 keys: 953 against 1025 us a token).
// The kernel boundaries are the only
// synchronisation.  pv_j is 512 bytes per head and block, half of what the
// block's K and V rows hold for the two heads, so the split pays while the
// launch is short of workgroups, not when a batch fills the chip
// (attn_split_batch).
#include "q3_attn_v.h"
#include "q3_device.h"
#include "q3_epi.h"
#include "q3_kernels.h"

namespace q3 {
namespace {

constexpr int kWaves = 4;   // blocks per workgroup (one per wave)
constexpr int kGrp = 2;     // query heads per KV head
constexpr float kFloor = -3.402823466e38f;  // the walk's first maximum (attention_gqa.h:418)

struct Unit {
  int row, split, kvh, nblk;
  uint32_t kv_len;
  const uint16_t *table;
};

// Workgroup id -> (KV head, sequence, 4-block run): ids with equal residues
// mod 8 run on one XCD, so the KV heads of a run (which share its page-table
// and scale lines) get ids with one residue.
__device__ __forceinline__ Unit make_unit(const SplitArgs &a) {
  const int id = static_cast<int>(blockIdx.x);
  const int t = id >> 3;
  const int u = (t / a.kv_heads) * 8 + (id & 7);
  Unit w;
  w.kvh = t % a.kv_heads;
  w.row = u % a.rows;
  w.split = u / a.rows;
  w.kv_len = a.row_pos ? static_cast<uint32_t>(a.row_pos[w.row]) + 1 : a.kv_len;
  w.nblk = static_cast<int>((w.kv_len + 31) / 32);
  w.table = a.row_pos ? a.table + static_cast<int64_t>(w.row) * a.ld_table : a.table;
  return w;
}

__global__ void __launch_bounds__(kWaves * 64) split_score_kernel(SplitArgs a) {
  __shared__ __align__(16) int8_t q8s[kGrp][HD];
  __shared__ __align__(16) int8_t knew[HD];
  __shared__ float qss[kGrp], ksnew;
  const Unit u = make_unit(a);
  if (u.split * kWaves >= u.nblk) return;
  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int blk = u.split * kWaves + wave;
  const int jb = min(blk, u.nblk - 1);
  const int j = jb * 32;
  const int pos0 = static_cast<int>(u.kv_len) - 1;
  const bool tail = (u.split + 1) * kWaves >= u.nblk;  // holds the new token's block
  // this wave's projection row: waves 0, 1 a query head each, 2 K, 3 V
  const int qh = u.kvh * kGrp + (wave & 1);
  const float *src = wave < kGrp  ? a.fq + static_cast<int64_t>(u.row) * a.ldq + qh * HD
                     : wave == 2 ? a.fk + static_cast<int64_t>(u.row) * a.ldk + u.kvh * HD
                                 : a.fv + static_cast<int64_t>(u.row) * a.ldk + u.kvh * HD;
  float t0 = src[lane], t1 = src[lane + 64];
  const float *nw = wave < kGrp ? a.nq : a.nk;
  const float w0 = nw[lane], w1 = nw[lane + 64];
  const float c = a.cos_t[static_cast<int64_t>(pos0) * 64 + lane];
  const float sn = a.sin_t[static_cast<int64_t>(pos0) * 64 + lane];
  // K rows and scales of the wave's block (keys past the last repeat it)
  const uint32_t page = u.table[static_cast<uint32_t>(j) / a.page_tokens];
  const uint32_t slot0 = static_cast<uint32_t>(j) % a.page_tokens;
  const int8_t *kb = a.k + page * a.page_bytes + slot0 * a.row_bytes + u.kvh * HD;
  const int8_t *ksb = reinterpret_cast<const int8_t *>(a.ks) + page * a.scale_page_bytes + slot0 * a.scale_row_bytes;
  const int last = pos0 - j;
  const int kg = lane >> 3, kb16 = 16 * (lane & 7);
  const int kcl = 8 * ((lane >> 1) & 3) + kg;  // key whose score the lane ends with
  int4 kw[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    kw[e] = *reinterpret_cast<const int4 *>(kb + min(8 * e + kg, last) * a.row_bytes + kb16);
  float kscale = reinterpret_cast<const float *>(ksb + min(kcl, last) * a.scale_row_bytes)[u.kvh];
  uint32_t npage = 0;
  if (tail) npage = u.table[static_cast<uint32_t>(pos0) / a.page_tokens];
  // ---- head epilogues (norm_rope_quant.h:17-86, group_gemm.h:173-193) ----
  if (wave < kGrp || tail) {
    if (wave != 3) head_norm_rope_regs(t0, t1, w0, w1, c, sn, a.inv_hd, true);
    const float scale = __fmul_rn(max64(fmaxf(fabsf(t0), fabsf(t1))), inv127());
    const int8_t q0 = static_cast<int8_t>(quant1(t0, scale));
    const int8_t q1 = static_cast<int8_t>(quant1(t1, scale));
    if (wave < kGrp) {
      q8s[wave][lane] = q0;
      q8s[wave][lane + 64] = q1;
      if (lane == 0) qss[wave] = scale;
      if (tail) {  // the int8 row for the record
        int8_t *row8 = a.q8 + static_cast<int64_t>(u.row) * a.ldq8 + qh * HD;
        row8[lane] = q0;
        row8[lane + 64] = q1;
        if (lane == 0) a.qs[static_cast<int64_t>(u.row) * a.ldqs + qh] = scale;
      }
    } else {
      if (wave == 2) {
        knew[lane] = q0;
        knew[lane + 64] = q1;
        if (lane == 0) ksnew = scale;
      }
      const uint32_t slot = static_cast<uint32_t>(pos0) % a.page_tokens;
      int8_t *row8 = (wave == 2 ? a.k : a.v) + npage * a.page_bytes + slot * a.row_bytes + u.kvh * HD;
      float *sp = reinterpret_cast<float *>(reinterpret_cast<int8_t *>(wave == 2 ? a.ks : a.vs) +
                                            npage * a.scale_page_bytes + slot * a.scale_row_bytes) + u.kvh;
      row8[lane] = q0;
      row8[lane + 64] = q1;
      if (lane == 0) *sp = scale;
    }
  }
  __syncthreads();
  if (blk >= u.nblk) return;
  if (pos0 < j + 32) {  // the new token's K row from LDS (its page slot may not be visible)
    const int4 kn = *reinterpret_cast<const int4 *>(knew + kb16);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (j + 8 * e + kg >= pos0) kw[e] = kn;
    if (j + kcl >= pos0) kscale = ksnew;
  }
  const int64_t ws0 = (static_cast<int64_t>(u.row) * a.heads + u.kvh * kGrp) * a.ldb + jb;
#pragma unroll
  for (int h = 0; h < kGrp; ++h) {
    const int4 q = *reinterpret_cast<const int4 *>(q8s[h] + kb16);
    int p[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p[e] = sdot4(q.x, kw[e].x, 0);
      p[e] = sdot4(q.y, kw[e].y, p[e]);
      p[e] = sdot4(q.z, kw[e].z, p[e]);
      p[e] = sdot4(q.w, kw[e].w, p[e]);
    }
    // exact int32 sums over the 8 lanes of a key, scattered over lane bits
    // 2, 1, 0 so that lanes 2m, 2m + 1 end with key kcl
    const bool b2 = lane & 4, b1 = lane & 2;
    int k0 = b2 ? p[2] : p[0], k1 = b2 ? p[3] : p[1];
    k0 += lane_xor<4>(b2 ? p[0] : p[2]);
    k1 += lane_xor<4>(b2 ? p[1] : p[3]);
    int acc = b1 ? k1 : k0;
    acc += lane_xor<2>(b1 ? k0 : k1);
    acc += lane_xor<1>(acc);
    float s = -INFINITY;
    if (j + kcl <= pos0) {
      s = __fmul_rn(static_cast<float>(acc), kscale);
      s = __fmul_rn(s, qss[h]);
      s = __fmul_rn(s, a.qk_scale);
    }
    const float bm = max64(s);
    const int64_t wb = ws0 + h * a.ldb;
    if ((lane & 1) == 0) a.ws_s[wb * 32 + kcl] = s;
    if (lane == 0) a.ws_bmax[wb] = bm;
  }
}

__global__ void __launch_bounds__(kWaves * 64) split_pv_kernel(SplitArgs a) {
  __shared__ uint64_t tab[32];
  __shared__ __align__(16) int8_t vst[kWaves][32 * HD];
  __shared__ __align__(16) int8_t p8s[kWaves][kGrp][32];
  const Unit u = make_unit(a);
  if (u.split * kWaves >= u.nblk) return;
  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int blk = u.split * kWaves + wave;
  const int jb = min(blk, u.nblk - 1);
  const int j = jb * 32;
  const int last = static_cast<int>(u.kv_len) - 1 - j;
  const uint32_t page = u.table[static_cast<uint32_t>(j) / a.page_tokens];
  const uint32_t slot0 = static_cast<uint32_t>(j) % a.page_tokens;
  const int8_t *vb = a.v + page * a.page_bytes + slot0 * a.row_bytes + u.kvh * HD;
  const int8_t *vsb = reinterpret_cast<const int8_t *>(a.vs) + page * a.scale_page_bytes + slot0 * a.scale_row_bytes;
  // the block's V rows into the wave's stage, then the score, scale and
  // block-maximum loads
  int8_t *st = vst[wave];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = 8 * e + (lane >> 3);
    lds_copy16(vb + min(r, last) * a.row_bytes + 16 * ((lane & 7) ^ vswz(r)), st + 1024 * e);
  }
  // lane = 32 h + key (scores), 32 h + block (maxima)
  const int c = lane & 31, h = lane >> 5;
  const int64_t wb = (static_cast<int64_t>(u.row) * a.heads + u.kvh * kGrp + h) * a.ldb;
  const float s = a.ws_s[(wb + jb) * 32 + c];
  const float vscale = reinterpret_cast<const float *>(vsb + min(c, last) * a.scale_row_bytes)[u.kvh];
  const float own = a.ws_bmax[wb + jb];
  // maximum of the blocks before this one (any order: scores are never NaN
  // nor -0, so the walk's select max is associative)
  float m = kFloor;
  for (int i = c; i < jb; i += 128) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = a.ws_bmax[wb + min(i + 32 * e, jb - 1)];
    m = fmaxf(m, fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])));
  }
  if (threadIdx.x == 0) stage_exp2_table(tab);
  wait_vmcnt<0>();  // the copies have landed
  __syncthreads();
  if (blk >= u.nblk) return;
  const float nmm = fmaxf(max32(m), own);
  float p = 0.0f, pv = 0.0f;
  if (c <= last) {
    p = exp_f32_le0_tab(__fsub_rn(s, nmm), tab);
    pv = __fmul_rn(p, vscale);
  }
  const float psum = tree_sum32(p);
  const float pm = __fmul_rn(max32(pv), inv127());
  p8s[wave][h][p8_pos(c)] = static_cast<int8_t>(quant1(pv, pm));
  if (c == 0) {
    a.ws_psum[wb + jb] = psum;
    a.ws_nmm[wb + jb] = nmm;
  }
  // P8.V (k_attn_decode.hip pv_mfma): A row m carries head m % 2's P8, so
  // result register q of every lane holds head q % 2, dim 16 t + lane % 16;
  // each 16-lane group stores two of the eight dim tiles
  const int tr_key = 16 * (((lane & 15) >> 1) >> 2) + 4 * (lane >> 4) + (((lane & 15) >> 1) & 3);
  const int tr_base = tr_key * HD + 8 * (lane & 1);
  const int tr_sw = vswz(tr_key);
  const float pm0 = lane_bcast<0>(pm), pm1 = lane_bcast<32>(pm);
  const long av = *reinterpret_cast<const long *>(p8s[wave][lane & 1] + 8 * (lane >> 4));
  const v4i_d z = {0, 0, 0, 0};
  v4i_d acc[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const v2i_d bt = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
        reinterpret_cast<lds_v2i_ptr_d>(to_lds(st + tr_base + ((t ^ tr_sw) << 4))));
    long bv;
    __builtin_memcpy(&bv, &bt, sizeof(bv));
    acc[t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bv, z, 0, 0, 0);
  }
  const int g = lane >> 4;
  float *dst = a.ws_pv + ((static_cast<int64_t>(u.row) * a.heads + u.kvh * kGrp) * a.ldb + jb) * HD;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    int i0 = acc[4 * q][0], i1 = acc[4 * q][1];
#pragma unroll
    for (int e = 1; e < 4; ++e) {
      i0 = g == e ? acc[4 * q + e][0] : i0;
      i1 = g == e ? acc[4 * q + e][1] : i1;
    }
    const int d = 64 * q + lane;
    dst[d] = __fmul_rn(static_cast<float>(i0), pm0);
    dst[static_cast<int64_t>(a.ldb) * HD + d] = __fmul_rn(static_cast<float>(i1), pm1);
  }
}

constexpr int kChainWaves = 8;
constexpr int kStage = 16;        // blocks per LDS stage (one instruction per wave)
constexpr int kStages = 8;        // stages in flight
constexpr int kChainBlocks = kStage * kStages;

__global__ void __launch_bounds__(kChainWaves * 64) split_chain_kernel(SplitArgs a) {
  __shared__ uint64_t tab[32];
  __shared__ __align__(16) float pvs[kChainBlocks][HD];
  __shared__ float amax[2];
  const int row = static_cast<int>(blockIdx.x) / a.heads;
  const int qh = static_cast<int>(blockIdx.x) % a.heads;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = wave_id();
  const uint32_t kv_len = a.row_pos ? static_cast<uint32_t>(a.row_pos[row]) + 1 : a.kv_len;
  const int nblk = static_cast<int>((kv_len + 31) / 32);
  const int64_t wb = (static_cast<int64_t>(row) * a.heads + qh) * a.ldb;
  if (tid == 0) stage_exp2_table(tab);
  float res = 0.0f, den = 0.0f;
  for (int b0 = 0; b0 < nblk; b0 += kChainBlocks) {
    const int nb = min(kChainBlocks, nblk - b0);
    // waves 0, 1: lane l's blocks b0 + 64 q + l: maximum, the one before, psum
    float nm[2], pm[2], ps[2], corr[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int jl = b0 + min(64 * q + lane, nb - 1);
      nm[q] = a.ws_nmm[wb + jl];
      pm[q] = a.ws_nmm[wb + max(jl - 1, 0)];
      if (jl == 0) pm[q] = kFloor;
      ps[q] = a.ws_psum[wb + jl];
    }
    // pv rows, 2 blocks per instruction (past the chunk: its last block);
    // stages past the chunk are not copied
#pragma unroll
    for (int e = 0; e < kStages; ++e) {
      if (kStage * e < nb) {
        const int j = kStage * e + 2 * wave;
        const int blk = b0 + min(j + (lane >> 5), nb - 1);
        lds_copy16(a.ws_pv + (wb + blk) * HD + 4 * (lane & 31), &pvs[j][0]);
      }
    }
    const bool full = nb > kStage * (kStages - 1);  // every stage was copied
    // stage e is complete once every wave's own copy of it has landed (one
    // wait for all of a partial chunk)
    static_for<kStages>([&](auto E) {
      constexpr int e = decltype(E)::value;
      if (kStage * e >= nb) return;
      if (full) {
        wait_vmcnt<kStages - 1 - e>();
        lds_barrier();
      } else if (e == 0) {
        wait_vmcnt<0>();
        lds_barrier();
      }
      if (wave < 2) {
        constexpr int q = kStage * e / 64, l0 = kStage * e % 64;
        if (l0 == 0) corr[q] = exp_f32_le0_tab(__fsub_rn(pm[q], nm[q]), tab);
        float pw[kStage];
#pragma unroll
        for (int i = 0; i < kStage; ++i) pw[i] = pvs[kStage * e + i][tid];
#pragma unroll
        for (int i = 0; i < kStage; ++i) {
          if (kStage * e + i < nb) {
            const float cr = lane_read(corr[q], l0 + i);
            den = __fadd_rn(__fmul_rn(den, cr), lane_read(ps[q], l0 + i));
            res = __fadd_rn(__fmul_rn(res, cr), pw[i]);
          }
        }
      }
    });
    if (b0 + kChainBlocks < nblk) {
      wait_vmcnt<0>();
      lds_barrier();  // the stages are free again
    }
  }
  // ---- epilogue: out = res * (1/den); per-head int8 quant (522-546) ----
  float out = 0.0f;
  if (wave < 2) {
    out = __fmul_rn(res, __fdiv_rn(1.0f, den));
    const float mx = max64(fabsf(out));
    if (lane == 0) amax[wave] = mx;
  }
  wait_vmcnt<0>();
  lds_barrier();
  if (wave < 2) {
    const float scale = __fmul_rn(fmaxf(amax[0], amax[1]), inv127());
    a.o8[static_cast<int64_t>(row) * a.ldo + qh * HD + tid] = static_cast<int8_t>(quant1(out, scale));
    if (tid == 0) a.os[static_cast<int64_t>(row) * a.ldos + qh] = scale;
  }
}

}  // namespace

bool attn_split_supported(const SplitArgs &a) {
  auto al16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (a.rows < 1 || a.kv_heads < 1 || a.heads != kGrp * a.kv_heads || a.max_blocks < 1 || a.ldb < a.max_blocks)
    return false;
  if (a.page_tokens % 32 || a.row_bytes % 16 || a.page_bytes % 16 || a.scale_row_bytes % 4 || !al16(a.k) || !al16(a.v))
    return false;
  if (!a.ws_s || !a.ws_bmax || !a.ws_nmm || !a.ws_psum || !a.ws_pv || !al16(a.ws_pv)) return false;
  return true;
}

// A batch takes the split when the single launch's serial walk of its longest
// row (~0.53 us per block past the first chunk) costs more than the split's
// work over all rows (~0.016 us per row and block) and its extra launches.
// Measured on the 28-layer decode step, us (single launch / split):
// 1 row x 384 keys 1127 / 1099, 1 x 2048 1942 / 1168, 5 x 700 1469 / 1306,
// 16 x 384 1339 / 1371, 16 x 2048 2210 / 1745, 24 x 700 1579 / 1560, 32 x
// 1024 1784 / 1789, 32 x 2048 2349 / 2217, 48 x 2048 2665 / 2795, 64 x 2048
// 2854 / 3308.
bool attn_split_batch(int64_t max_blocks, int64_t sum_blocks) {
  return max_blocks >= 12 && 36 * max_blocks > sum_blocks + 250;
}

hipError_t launch_attn_split(const SplitArgs &a, hipStream_t s) {
  if (!attn_split_supported(a)) return hipErrorInvalidValue;
  const int64_t units = static_cast<int64_t>(a.rows) * ((a.max_blocks + kWaves - 1) / kWaves);
  const int64_t grid = (units + 7) / 8 * 8 * a.kv_heads;
  if (grid >= (int64_t{1} << 31)) return hipErrorInvalidValue;
  Q3_LAUNCH(split_score_kernel, dim3(static_cast<unsigned>(grid)), dim3(kWaves * 64), 0, s, a);
  Q3_LAUNCH(split_pv_kernel, dim3(static_cast<unsigned>(grid)), dim3(kWaves * 64), 0, s, a);
  Q3_LAUNCH(split_chain_kernel, dim3(static_cast<unsigned>(a.rows * a.heads)), dim3(kChainWaves * 64), 0, s, a);
  return hipGetLastError();
}

}  // namespace q3
