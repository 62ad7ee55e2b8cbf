// GQA flash-attention forward for small grids (hot-path row R1), gfx950.
//
// Same results as fwd_kernel (gfa_fwd.hip) by another split of the work. fwd_kernel gives every
// wave 32 query rows and all of their keys: it reads each K / V tile once per 128 query rows,
// but a short prompt then launches a few dozen workgroups for 256 CUs and its time is the
// longest row's serial walk over the keys. Here a workgroup owns 32 query rows of one head
// and its four waves split the KEYS: four times the workgroups, a quarter of the serial walk.
//  * A wave (D <= 256) or a wave pair (D = 512, each wave over one half of the head dim) is a
//    key group: group g takes the key tiles t_lo + g, t_lo + g + NG, ... with its own
//    softmax reference, row sum and O^T accumulator, exactly as a wave of fwd_kernel does, and
//    the groups' results are combined once, at the end, through LDS in fp32.
//  * A wave's tiles are private, so the loop has no workgroup barrier at D <= 256; at D = 512 the
//    two waves of a pair add their halves of S once per tile (one barrier).
//  * A tile is 8192 elements of K and of V per wave (32 keys at a width of 256, 64 at 128, 128 at
//    64), in two cells each of 32 rows x 128 columns (64 x 64 at D = 64; 8 KB, one LDS object per
//    cell). A cell is consumed by eight products; its refill (the next tile's cell, eight 1 KB
//    direct global->LDS copies) is issued one copy per product right behind it, so the copies
//    run most of a tile ahead of their use out of a single-buffered tile. The copies' row
//    pieces are 256 bytes: with 128-byte ones (cells of 64 columns) the kernel took 3-6% longer at
//    D >= 256 (8:1 D=512 N=2048 causal 70.4 -> 66.4 us, 8:4 D=256 N=700 13.9 -> 12.8 us).
// Bound: the longest row's walk by one wave per SIMD. Every wave reads its own K / V from L2, 32 rows
// of queries per tile byte (128 in fwd_kernel), so at best (64 B per CU and clock) the copies take
// twice the products' time; at D=512 8:1 N=1024 a CU gets about 30 of them over the kernel (36 us
// without a mask, 33 causal with half the bytes in all but the same longest row), matrix cores
// 16% and 9% busy. The host takes this kernel where the 128-row grid leaves CUs idle (gfa_api.hip).
#include "gfa_common.h"
#include "gfa_params.h"
#include "gfa_launch.h"

namespace gfa {

namespace {

// Wait until at most N of this wave's vector-memory operations (tile copies) are outstanding.
template <int N>
__device__ __forceinline__ void wait_copies() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Copies cells (4096 elements: 4096 / CW rows x CW columns of a row-major 16-bit slice) into LDS: row r at
// byte 2 CW r, 16-byte chunk c at chunk position c ^ swz<CW>(r). Eight instructions of whole row
// pieces.
template <int CW>
struct CellLoader {
  static constexpr int LPR = CW / 8;    // lanes per row piece
  static constexpr int RPI = 64 / LPR;  // rows per instruction
  static constexpr int NV = 16 / RPI;   // the swizzle repeats every 16 rows
  __amdgpu_buffer_rsrc_t rsrc;
  unsigned voff[NV];
  unsigned stride_b;
  __device__ __forceinline__ void init(const uint16_t* base, int64_t row_stride, int n_rows, int row_elems, int lane) {
    stride_b = (unsigned)(row_stride * 2);
    rsrc = slice_rsrc(base, row_stride, n_rows, row_elems);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int row = RPI * i + lane / LPR;
      voff[i] = (lane / LPR) * stride_b + (unsigned)(((lane % LPR) ^ swz<CW>(row)) << 4);
    }
  }
  // Instruction i (< 8) of the cell at rows row0 .., columns from byte col_b of the row.
  __device__ __forceinline__ void load_part(int i, int row0, int col_b, char GFA_LDS* cell) const {
    const unsigned soff = (unsigned)(row0 + RPI * i) * stride_b + (unsigned)col_b;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (void GFA_LDS*)(cell + i * 1024), 16, voff[i % NV], soff, 0, 0);
  }
};

}  // namespace

template <int D, bool IS_BF16, bool SEG, bool CAP, bool DROP>
__global__ __launch_bounds__(256, 1) void fwd_rows_kernel(const FwdParams p) {
  constexpr int SD = D == 512 ? 2 : 1;  // waves per key group, each over DW columns of the head dim
  constexpr int NG = 4 / SD;            // key groups
  constexpr int DW = D / SD;
  constexpr int BKV = 8192 / DW;        // keys per tile
  constexpr int KT = DW / 16;
  constexpr int DB = DW / 32;
  constexpr int SB = BKV / 32;
  constexpr int CW = DW < 128 ? DW : 128;  // cell: CR rows x CW columns
  constexpr int CR = 4096 / CW;
  constexpr int CG = DW / CW;           // cells side by side
  constexpr int CELL = 8192;
  constexpr int PF = 4;                 // LDS read-ahead, in products
  constexpr float kMargin = IS_BF16 ? 64.0f : 15.0f;      // as fwd_kernel
  constexpr float kMaxRowSum = 18446744073709551616.0f;
  constexpr bool LAZY = IS_BF16;
  static_assert(SB * KT == 16 && SB * 2 * DB == 16 && BKV / CR * CG == 2, "16 products and two cells per phase");
  static_assert(PF == 4, "the copy counts below assume a read-ahead of half a cell");

  // One LDS object per cell (the compiler tells a read of one cell from the copies in flight into
  // the others), each with an 8 KB block per wave.
  __shared__ __attribute__((aligned(1024))) char k0_lds[4 * CELL], k1_lds[4 * CELL];
  __shared__ __attribute__((aligned(1024))) char v0_lds[4 * CELL], v1_lds[4 * CELL];
  // SD = 2: the pairs' S halves, double buffered (4 KB per wave). After the loop: row statistics.
  constexpr int PX = SD == 2 ? 2 * 4 * 4096 : 1024;
  __shared__ __attribute__((aligned(1024))) char x_lds[PX];
  char GFA_LDS* const xl = (char GFA_LDS*)x_lds;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wave / SD;
  const int dh = wave % SD;
  const int h = lane >> 5;
  const int l32 = lane & 31;
  auto kcell = [&](int c, int w) __attribute__((always_inline)) {
    return (c == 0 ? (char GFA_LDS*)k0_lds : (char GFA_LDS*)k1_lds) + w * CELL;
  };
  auto vcell = [&](int c, int w) __attribute__((always_inline)) {
    return (c == 0 ? (char GFA_LDS*)v0_lds : (char GFA_LDS*)v1_lds) + w * CELL;
  };

  // ---- workgroup -> (b, head, 32-row query block); the R heads of a KV head side by side on one
  // XCD (they read the same K / V), under causal masking the longest rows first ----
  int lid = xcd_remap((int)blockIdx.x, p.g.nblocks, p.R);
  const int head_r = lid % p.R;
  lid /= p.R;
  const int kvh = lid % p.Hkv;
  lid /= p.Hkv;
  const int b = lid % p.B;
  lid /= p.B;
  const int q0 = 32 * (p.causal ? (p.g.n_qsb - 1 - lid) : lid);
  const int head = kvh * p.R + head_r;
  const int q_hi = min(p.N, q0 + 32);

  const bool swa = p.causal && p.window > 0;
  int k_lo = 0, k_hi = p.N;
  int all_lo = 0, all_hi = p.N;  // keys every query of the block sees
  if (p.causal) {
    k_hi = q_hi;
    all_hi = min(p.N, q0 + 1);
    if (swa) {
      k_lo = max(0, q0 - p.window + 1);
      all_lo = q0 + 31 - p.window + 1;
    }
  }
  const int q = q0 + l32;
  const int qr = min(q, p.N - 1);
  VisRange vis_seg{};
  if constexpr (SEG) {
    const int* slo = p.seg_lo + (int64_t)b * p.N;
    const int* shi = p.seg_hi + (int64_t)b * p.N;
    k_lo = max(k_lo, clamp_n(slo[q0], p.N));
    k_hi = min(k_hi, clamp_n(shi[q_hi - 1], p.N));
    all_lo = max(all_lo, clamp_n(slo[q_hi - 1], p.N));
    all_hi = min(all_hi, clamp_n(shi[q0], p.N));
    vis_seg = intersect(keys_of_query(q, p.N, p.causal, p.window), clamp_n(slo[qr], p.N), clamp_n(shi[qr], p.N));
  }
  const int t_lo = k_lo / BKV;
  const int t_hi = k_hi > k_lo ? (k_hi + BKV - 1) / BKV : t_lo;
  // Tiles of this group. SD = 2: every group runs the workgroup's longest count (the pair barrier is
  // a workgroup barrier); a group's tile past t_hi is fully masked and copies nothing.
  const int steps = SD == 2 ? (t_hi - t_lo + NG - 1) / NG : max(0, (t_hi - t_lo - grp + NG - 1) / NG);

  CellLoader<CW> kload, vload;
  kload.init(p.k + (int64_t)b * p.kv.sb + (int64_t)kvh * p.kv.sh, p.kv.sn, p.N, D, lane);
  vload.init(p.v + (int64_t)b * p.vv.sb + (int64_t)kvh * p.vv.sh, p.vv.sn, p.N, D, lane);
  // Copy instruction i of cell c of the tile at row0.
  auto kcopy = [&](int c, int i, int row0) __attribute__((always_inline)) {
    kload.load_part(i, row0 + CR * (c / CG), 2 * CW * (c % CG) + 2 * DW * dh, kcell(c, wave));
  };
  auto vcopy = [&](int c, int i, int row0) __attribute__((always_inline)) {
    vload.load_part(i, row0 + CR * (c / CG), 2 * CW * (c % CG) + 2 * DW * dh, vcell(c, wave));
  };
  // First row of step s's tile; rows past the sequence end (no such tile) copy zeros, no memory read.
  auto row_of = [&](int s) __attribute__((always_inline)) {
    const int t = t_lo + s * NG + grp;
    return t < t_hi ? t * BKV : p.N;
  };

  // ---- Q fragments (B operand of S^T = K Q^T) ----
  i16x8 qf[KT];
  {
    const uint16_t* qp = p.q + (int64_t)b * p.qv.sb + (int64_t)head * p.qv.sh + (int64_t)qr * p.qv.sn + DW * dh + 8 * h;
#pragma unroll
    for (int kk = 0; kk < KT; ++kk) qf[kk] = *reinterpret_cast<const i16x8*>(qp + 16 * kk);
  }

  // Per-lane LDS offsets inside a cell: K row l32 at chunk 2 kk + h; V read transposed (rows 4h + t/4
  // and 8 further, column block 0). As kstep_off / mma_tr_accumulate_b at D = CW.
  const int koff0 = l32 * (2 * CW) + ((h ^ swz<CW>(l32)) << 4);
  int voff0;
  {
    const int t16 = lane & 15;
    const int rA = 4 * h + (t16 >> 2);
    const int c = 2 * ((lane >> 4) & 1) + ((t16 >> 1) & 1);
    voff0 = rA * (2 * CW) + ((c ^ swz<CW>(rA)) << 4) + (t16 & 1) * 8;
  }
  // A operand of S product i (key block i / KT, k-step i % KT; cell i / 8) and of PV product i: cell
  // i / 8, then the k-steps of its rows, then its column blocks.
  auto kfrag = [&](int i) __attribute__((always_inline)) {
    const int kk = i % (CW / 16), rb = (i & 7) / (CW / 16);  // k-step, 32-row block inside the cell
    return lds_read16(kcell(i >> 3, wave), (koff0 ^ (kk << 5)) + rb * 32 * (2 * CW));
  };
  constexpr int CB = CW / 32;  // column blocks per cell
  auto vfrag = [&](int i) __attribute__((always_inline)) {
    const int a = voff0 ^ ((i % CB) << 6);
    return tr_frag(vcell(i >> 3, wave), a, (a ^ 32) + 16 * CW, ((i & 7) / CB) * 16 * (2 * CW));
  };

  f32x16 acc[DB];
  float m_ref = kNegBig, m_seen = kNegBig, l_run = 0.f;
  bool ovf = false;
  const float xs = CAP ? p.cap.cap_log2 : p.scale_log2;
  const unsigned drow = DROP ? drop_row(p.drop.seed_lo, p.drop.seed_hi, b * p.Hq + head, q) : 0u;

  // S^T of step s's tile, masked (CAP: tanh of it). `behind(i)` issues a copy behind product i.
  auto scores = [&](int s, f32x16 (&sc)[SB], auto&& behind) __attribute__((always_inline)) {
    i16x8 a[PF];
#pragma unroll
    for (int i = 0; i < PF; ++i) a[i] = kfrag(i);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const i16x8 cur = a[i % PF];
      if (i + PF < 16) {
        if (i + PF == 8) wait_copies<12>();
        a[i % PF] = kfrag(i + PF);
      }
      // in VGPRs (O^T is pinned to AGPRs; see mma32_vgpr)
      if (i % KT == 0) {
        mma32_vgpr<IS_BF16, true>(sc[i / KT], cur, qf[i % KT]);
      } else {
        mma32_vgpr<IS_BF16, false>(sc[i / KT], cur, qf[i % KT]);
      }
      behind(i);
    }
#pragma unroll
    for (int sb = 0; sb < SB; ++sb) mfma_result_fence(sc[sb]);
    if constexpr (SD == 2) {
      // The pair's halves of S: both waves hold own + partner (the same sum in both).
      char GFA_LDS* const mine = xl + (s & 1) * (4 * 4096) + wave * 4096 + lane * 16;
      const char GFA_LDS* const other = xl + (s & 1) * (4 * 4096) + (wave ^ 1) * 4096 + lane * 16;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4 GFA_LDS*>(mine + j * 1024) =
            f32x4{sc[0][4 * j], sc[0][4 * j + 1], sc[0][4 * j + 2], sc[0][4 * j + 3]};
      barrier_lds();
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 w = *reinterpret_cast<const f32x4 GFA_LDS*>(other + j * 1024);
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[0][4 * j + e] += w[e];
      }
    }
    if constexpr (CAP) {
#pragma unroll
      for (int sb = 0; sb < SB; ++sb) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[sb][r] = cap_tanh(sc[sb][r] * p.cap.cap_a);
      }
    }
    const int k0 = (t_lo + s * NG + grp) * BKV;
    if (!(k0 + BKV <= all_hi && k0 >= all_lo)) {
      const VisRange vis = SEG ? vis_seg : keys_of_query(q, p.N, p.causal, p.window);
#pragma unroll
      for (int sb = 0; sb < SB; ++sb) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = k0 + sb * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
          sc[sb][r] = vis.has(key) ? sc[sb][r] : -INFINITY;
        }
      }
    }
  };
  auto row_max = [&](const f32x16 (&sc)[SB]) __attribute__((always_inline)) {
    float m = -INFINITY;
#pragma unroll
    for (int sb = 0; sb < SB; ++sb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) m = fmaxf(m, sc[sb][r]);
    }
    return halves_max(m) * xs;
  };

  // One pass over the group's tiles. Cells are consumed in the order K0, K1, V0, V1; behind a cell's
  // products go the eight copies that refill the cell before it with the next tile (V1 behind K0,
  // K1 behind V0). Before a phase's first read the copies issued after its first cell are two
  // cells' (16 instructions), before the first read of its second cell (PF products ahead) one and
  // a half's (12).
  auto run_pass = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < DB; ++i) acc[i] = f32x16{};
    l_run = 0.f;
    int row = row_of(0);
    if (steps > 0) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (c < 2) {
            kcopy(c, i, row);
          } else {
            vcopy(0, i, row);
          }
        }
      }
      // The Q loads complete here, ahead of the copies in flight (left to the loop's first use, the
      // compiler drains every copy before the loop).
#pragma unroll
      for (int kk = 0; kk < KT; ++kk) pin_vgpr(qf[kk]);
    }
    for (int s = 0; s < steps; ++s) {
      const int next = row_of(s + 1);
      f32x16 sc[SB];
      wait_copies<16>();
      scores(s, sc, [&](int i) __attribute__((always_inline)) {
        if (i < 8) {
          vcopy(1, i, row);
        } else {
          kcopy(0, i - 8, next);
        }
      });
      if (!LAZY || __builtin_amdgcn_ballot_w64(m_ref == kNegBig) != 0) {
        const float mt = row_max(sc);
        m_ref = (m_ref == kNegBig && mt > kNegBig) ? mt : m_ref;
        if constexpr (!LAZY) {
          ovf = ovf || (mt > m_ref + kMargin);
          m_seen = fmaxf(m_seen, mt);
        }
      }
      i16x8 pb[2 * SB];
#pragma unroll
      for (int sb = 0; sb < SB; ++sb) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float pv = fast_exp2(sc[sb][r] * xs - m_ref);
          l_run += pv;
          float pk = pv;
          if constexpr (DROP) {
            const int key = (t_lo + s * NG + grp) * BKV + sb * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
            pk = drop_keep(drow, key, p.drop.thresh) ? pv : 0.f;
          }
          pb[sb * 2 + (r >> 3)][r & 7] = to16<IS_BF16>(pk);
        }
      }
      wait_copies<16>();
      i16x8 a[PF];
#pragma unroll
      for (int i = 0; i < PF; ++i) a[i] = vfrag(i);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int rb = (i >> 3) / CG, cg = (i >> 3) % CG;
        const int ks = CR / 16 * rb + (i & 7) / CB, db = CB * cg + i % CB;
        const i16x8 cur = a[i % PF];
        if (i + PF < 16) {
          if (i + PF == 8) wait_copies<12>();
          a[i % PF] = vfrag(i + PF);
        }
        acc[db] = mma32<IS_BF16>(cur, pb[ks], acc[db]);
        if (i < 8) {
          kcopy(1, i, next);
        } else {
          vcopy(0, i - 8, next);
        }
      }
#pragma unroll
      for (int i = 0; i < DB; ++i) pin_agpr(acc[i]);
      row = next;
    }
    drain_tile_copies();
  };
  run_pass();

  // ---- combine the groups ----
  // Row statistics of every group: [wave][m_ref | row sum][32 rows]. A sum past the limit (fp16: any
  // score past the reference's margin) makes the whole workgroup redo its rows with the exact
  // row max; every wave reads the same statistics and takes the same decision.
  float GFA_LDS* const st = (float GFA_LDS*)xl;
  float m_all[NG], l_all[NG];
  auto exchange = [&]() __attribute__((always_inline)) {
    barrier_lds();  // every wave is done with the exchange area
    const float l_row = halves_sum(l_run);
    if (h == 0) {
      st[wave * 64 + l32] = m_ref;
      st[wave * 64 + 32 + l32] = ovf ? INFINITY : l_row;
    }
    barrier_lds();
    bool over = false;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      m_all[g] = st[g * SD * 64 + l32];
      l_all[g] = st[g * SD * 64 + 32 + l32];
      over = over || l_all[g] > kMaxRowSum;
    }
    return over;
  };
  const bool over = exchange();
  if (__any(over)) {
    barrier_lds();
    if constexpr (LAZY) {
      // exact row max of the group's keys: the S^T products alone, one tile at a time
      for (int s = 0; s < steps; ++s) {
        const int row = row_of(s);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
          for (int i = 0; i < 8; ++i) kcopy(c, i, row);
        }
        wait_copies<0>();
        f32x16 sc[SB];
        scores(s, sc, [](int) {});
        m_seen = fmaxf(m_seen, row_max(sc));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
      barrier_lds();
    }
    m_ref = m_seen;
    ovf = false;
    run_pass();
    // (with the exact row max no score is past the margin)
    if constexpr (!LAZY) ovf = false;
    exchange();
  }
  float m_tot = kNegBig;
#pragma unroll
  for (int g = 0; g < NG; ++g) m_tot = fmaxf(m_tot, m_all[g]);
  float l_tot = 0.f;
#pragma unroll
  for (int g = 0; g < NG; ++g) l_tot += l_all[g] * fast_exp2(m_all[g] - m_tot);
  // a row that sees no key (empty segment): O = 0; DROP: kept P scaled by 1 / (1 - p)
  const float f = l_tot > 0.f ? fast_exp2(m_ref - m_tot) * (DROP ? p.drop.inv_keep : 1.0f) / l_tot : 0.f;
  if (p.store_lse && wave == 0 && h == 0 && q < p.N)
    p.lse[((int64_t)b * p.Hq + head) * p.lse_ld + q] = (m_tot + __log2f(l_tot)) * kLn2;

  // This wave's normalised O (fp32) into its own cells: two 4 KB accumulator blocks db per cell (K0,
  // K1, V0, V1), row r at byte 128 r, 16-byte chunk c (4 columns) at c ^ ((r >> 1) & 7).
  const int ln = opaque(lane);
  const int r32 = ln & 31;
  auto cell = [&](int db, int w) __attribute__((always_inline)) {
    return (db < 4 ? kcell(db >> 1, w) : vcell((db >> 1) - 2, w)) + (db & 1) * 4096;
  };
#pragma unroll
  for (int db = 0; db < DB; ++db) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 o4 = {acc[db][4 * g] * f, acc[db][4 * g + 1] * f, acc[db][4 * g + 2] * f, acc[db][4 * g + 3] * f};
      *reinterpret_cast<f32x4 GFA_LDS*>(cell(db, wave) + r32 * 128 + (((2 * g + (ln >> 5)) ^ ((r32 >> 1) & 7)) << 4)) = o4;
    }
  }
  barrier_lds();
  // Each wave sums and stores a share of the rows (of its head-dim half): rows 32 / NG * grp .., 8
  // rows x 64 columns per instruction, 16 bytes per lane, non-temporally (written once).
  uint16_t* const ob = p.o + (int64_t)b * p.ov.sb + (int64_t)head * p.ov.sh + DW * dh;
#pragma unroll
  for (int i = 0; i < 32 / NG / 8; ++i) {
    const int r = grp * (32 / NG) + 8 * i + (ln >> 3);
    const int sw = (r >> 1) & 7;
    const int c0 = 2 * (ln & 3);
#pragma unroll
    for (int j = 0; j < DW / 64; ++j) {
      f32x4 lo{}, hi{};
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        // columns 64 j + 32 ((ln >> 2) & 1) + 8 (ln & 3) ..: block 2 j or 2 j + 1, chunks c0, c0 + 1
        const int w = g * SD + dh;
        const char GFA_LDS* const src = ((ln >> 2) & 1) ? cell(2 * j + 1, w) : cell(2 * j, w);
        lo += *reinterpret_cast<const f32x4 GFA_LDS*>(src + r * 128 + ((c0 ^ sw) << 4));
        hi += *reinterpret_cast<const f32x4 GFA_LDS*>(src + r * 128 + (((c0 + 1) ^ sw) << 4));
      }
      i16x8 o8;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o8[e] = to16<IS_BF16>(lo[e]);
        o8[4 + e] = to16<IS_BF16>(hi[e]);
      }
      if (q0 + r < p.N)
        __builtin_nontemporal_store(o8, reinterpret_cast<i16x8*>(ob + (int64_t)(q0 + r) * p.ov.sn + 64 * j + 8 * (ln & 7)));
    }
  }
}

// Explicit instantiations of every built variant (device code and host launch stubs).
#define GFA_ROWS_INST(DD, CC, XX)                                                     \
  template __global__ void fwd_rows_kernel<DD, true, false, CC, XX>(const FwdParams);  \
  template __global__ void fwd_rows_kernel<DD, false, false, CC, XX>(const FwdParams); \
  template __global__ void fwd_rows_kernel<DD, true, true, CC, XX>(const FwdParams);   \
  template __global__ void fwd_rows_kernel<DD, false, true, CC, XX>(const FwdParams);
#define GFA_ROWS_INST_D(DD)       \
  GFA_ROWS_INST(DD, false, false) \
  GFA_ROWS_INST(DD, true, false)  \
  GFA_ROWS_INST(DD, false, true)
GFA_ROWS_INST_D(512)
GFA_ROWS_INST_D(256)
GFA_ROWS_INST_D(128)
GFA_ROWS_INST_D(64)
#undef GFA_ROWS_INST_D
#undef GFA_ROWS_INST

template <int D, bool IS_BF16, bool CAP, bool DROP>
static hipError_t launch_rows_t(const FwdParams& p, hipStream_t stream) {
  if (p.seg_lo != nullptr) {
    hipLaunchKernelGGL((fwd_rows_kernel<D, IS_BF16, true, CAP, DROP>), dim3(p.g.nblocks), dim3(256), 0, stream, p);
  } else {
    hipLaunchKernelGGL((fwd_rows_kernel<D, IS_BF16, false, CAP, DROP>), dim3(p.g.nblocks), dim3(256), 0, stream, p);
  }
  return hipGetLastError();
}

hipError_t launch_fwd_rows(const FwdParams& p, int D, bool bf16, bool cap, bool drop, hipStream_t stream) {
#define GFA_ROWS_CASE(DD, CC, XX)                                                       \
  if (D == DD && cap == CC && drop == XX) {                                             \
    return bf16 ? launch_rows_t<DD, true, CC, XX>(p, stream) : launch_rows_t<DD, false, CC, XX>(p, stream); \
  }
#define GFA_ROWS_D(DD)          \
  GFA_ROWS_CASE(DD, false, false) \
  GFA_ROWS_CASE(DD, true, false)  \
  GFA_ROWS_CASE(DD, false, true)
  GFA_ROWS_D(512)
  GFA_ROWS_D(256)
  GFA_ROWS_D(128)
  GFA_ROWS_D(64)
#undef GFA_ROWS_D
#undef GFA_ROWS_CASE
  return hipErrorInvalidValue;
}

}  // namespace gfa
