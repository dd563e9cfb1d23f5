// bsg_rows.hpp — kind 8, the GEMM kernel for batches of more than 64 rows.
#pragma once

#include "bsg_device.hpp"

namespace {

// One stage of an LDS ring, PIECES KiB, as a variable of its own: the compiler makes every LDS read
// wait for the last load it knows to target the same variable, so with all stages in one array each
// read would also wait for the loads just issued for the stages behind it (vmcnt(0) per block).
template <int PIECES, int STAGE>
__device__ __forceinline__ u32x4* ring_stage() {
  __shared__ __attribute__((aligned(16))) u32x4 s_stage[PIECES * 64];
  return s_stage;
}

// Kind 8 ("rows"): one work-group = BTT*16 batch rows x nv <= NSUB 16-column subtiles, nv from
// vt_columns.  At these batches what a compute unit takes in bounds the launch, and that is
// (rows + columns of its tile) x 128 bytes per block: 128 rows x up to 96 columns over 256 compute
// units is near the square that minimises it, where 64-row groups re-read every weight once per
// 64 rows.  Both operands of a block arrive by 16-byte-per-lane loads straight into LDS, each byte
// once per work-group, in a ring of DEPTH stages: wave w brings pieces w, w + NW, ... (1 KiB each;
// pieces past the tile's load zeros), so a stage is the same count of loads in every wave and its
// arrival is one wait by count and one barrier.  The waves are row halves x channel halves: each
// reads its rows' activation pieces and every weight piece of its channel half, and the channel
// halves meet in LDS at the end, in the ring's storage.
template <typename T, int BTT, int NSUB, int RW, int DEPTH, int SEL>
__global__ __launch_bounds__(128 * RW) void bsg_gemm_rows_kernel(GemmParams p) {
  constexpr int NW = 2 * RW;
  constexpr int NT = 64 * NW;
  constexpr int RT = BTT / RW;                    // row tiles per wave
  constexpr int XP = 2 * BTT;                     // activation pieces per block: row tile x channel half
  constexpr int LX = XP / NW;                     // ... per wave
  constexpr int LW = (2 * NSUB + NW - 1) / NW;    // weight pieces per wave (the last may be past the tile)
  constexpr int L = LX + LW;
  constexpr int PIECES = L * NW;
  static_assert(DEPTH % 2 == 0, "the register sets alternate with the stages");
  static_assert(RT % 2 == 0, "each channel half stores half of the row tiles");
  static_assert(XP % NW == 0 && BTT % RW == 0, "every wave loads whole pieces");
  constexpr int RF = RT * NSUB;                   // output fragments per row part
  static_assert(RF <= PIECES && RW <= DEPTH, "each row part's halves meet in a stage of their own");
  __shared__ __attribute__((aligned(16))) int s_ids[BSG_MAX_NBLK];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = w & 1, rw = w >> 1;  // this wave's channel half and row part
  // Row groups of one column group are neighbours in the order that tile_of_group gives an XCD, so
  // the second read of a weight line finds it in that XCD's L2.
  int lid, unused;
  tile_of_group(1, &lid, &unused);
  const int yg = p.n_tiles > 0 ? (int)(gridDim.x / (unsigned)p.n_tiles) : 1;
  const int tile = lid / yg;
  const int y0 = (lid - tile * yg) * (16 * BTT);
  int st, nv;
  vt_columns(tile, p.n_tiles, p.npad >> 4, &st, &nv);
  BSG_TL_DECL
  BSG_TL(0);

  const int na = stage_block_list<NT, SEL>(p, s_ids, list_entry_of_thread<SEL>(p));
  BSG_TL(1);

  const int blk_bytes = p.npad * 128;
  // Activation pieces as in kind 7: lane 4q + c loads row q, 16-byte chunk (c - f(q)) % 4 of a
  // 32-channel half, and lane m reads (row m % 16, chunk m / 16) back at 4r + (chunk + f(r)) % 4,
  // f(r) = r/2 + r/8, so that consecutive lanes hit distinct banks.
  const int xq = lane >> 2;
  auto rot = [](int r) { return ((r >> 1) + (r >> 3)) & 3; };
  int xoff[LX];
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int pc = w + NW * i;  // row tile pc / 2, channel half pc % 2
    const int row = y0 + 16 * (pc >> 1) + xq;
    xoff[i] = row < p.bt ? row * (int)p.ldx * 2 : kOOB;
  }
  const int xcol = 8 * (((lane & 3) - rot(xq)) & 3) + 32 * h;  // NW is even: a wave's pieces are all of half w % 2
  const int rd_pos = 4 * (lane & 15) + (((lane >> 4) + rot(lane & 15)) & 3);
  int woff[LW];
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int pc = w + NW * i;  // subtile pc / 2, channel half pc % 2: consecutive KiBs of the packed block
    woff[i] = pc < 2 * nv ? lane * 16 + st * 2048 + pc * 1024 : kOOB;
  }

  f32x4 acc[RT][NSUB];
#pragma unroll
  for (int bi = 0; bi < RT; ++bi)
#pragma unroll
    for (int s = 0; s < NSUB; ++s) acc[bi][s] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Stage d takes list entry t (none past the list: empty resources load zeros).
  // The entry's id is read one slot ahead, so no load waits for LDS.
  int next_id = 0;
  auto fetch_id = [&](int t) {
    const int id = s_ids[t < na ? t : 0];
    next_id = t < na ? id : -1;
  };
  auto issue = [&](auto dd, int t) {
    u32x4* const ring = ring_stage<PIECES, decltype(dd)::value>();
    const int blk = __builtin_amdgcn_readfirstlane(next_id);
    fetch_id(t + 1);
    const bool ok = blk >= 0 && blk < p.nblk;
    const char* wb = (const char*)p.wp + (size_t)(ok ? blk : 0) * (size_t)blk_bytes;
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(wb, ok ? blk_bytes : 0);
    const __amdgpu_buffer_rsrc_t xb = make_rsrc(p.x, ok ? p.x_bytes : 0);
    const int col = (ok ? blk : 0) * 64 + xcol;
    // Out-of-range lanes get the offset's top bit by arithmetic: a select here becomes a branch
    // around the load, and the count of loads that arrive() waits by would no longer hold.
    const int past = ((p.K - 1 - col) >> 31) & kOOB;
#pragma unroll
    for (int i = 0; i < LW; ++i) ld16_lds(wr, ring + (XP + w + NW * i) * 64, woff[i]);
#pragma unroll
    for (int i = 0; i < LX; ++i)
      ld16_lds(xb, ring + (w + NW * i) * 64, (xoff[i] + col * 2) | past);
  };
  // This wave's fragments of stage d, read one slot ahead of their MFMAs (two register sets).
  u32x4 xv[2][RT], wv[2][NSUB];
  auto read = [&](auto dd) {
    constexpr int d = decltype(dd)::value;
    const u32x4* const ring = ring_stage<PIECES, d>();
#pragma unroll
    for (int s = 0; s < NSUB; ++s) wv[d & 1][s] = ring[(XP + 2 * s + h) * 64 + lane];
#pragma unroll
    for (int bi = 0; bi < RT; ++bi) xv[d & 1][bi] = ring[(2 * (rw * RT + bi) + h) * 64 + rd_pos];
  };
  auto compute = [&](auto dd) {
    constexpr int d = decltype(dd)::value;
#pragma unroll
    for (int bi = 0; bi < RT; ++bi)
#pragma unroll
      for (int s = 0; s < NSUB; ++s) acc[bi][s] = Elem<T>::mfma(wv[d & 1][s], xv[d & 1][bi], acc[bi][s]);
  };
  // All but the newest `later` stages have arrived in LDS for every wave, and every wave's reads so
  // far have returned, so the stage it read last may be loaded again.
  auto arrive = [&](auto later) {
    vmem_wait<decltype(later)::value * L>();
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // Slot t: stage t + 1 arrives, stage t (read in the slot before) is refilled with block t + DEPTH,
  // and block t's MFMAs run under the LDS reads of block t + 1.
  if (na > 0) {
    fetch_id(0);
    static_for<DEPTH>([&](auto dd) { issue(dd, decltype(dd)::value); });
    arrive(std::integral_constant<int, DEPTH - 1>{});
    read(std::integral_constant<int, 0>{});
    // na rounded up to whole passes of the ring; the slots past the list multiply zeros
    for (int t0 = 0; t0 < na; t0 += DEPTH) {
      static_for<DEPTH>([&](auto dd) {
        constexpr int d = decltype(dd)::value;
        arrive(std::integral_constant<int, DEPTH - 2>{});
        issue(dd, t0 + d + DEPTH);
        __builtin_amdgcn_sched_barrier(0);
        read(std::integral_constant<int, (d + 1) % DEPTH>{});
        // left free, the scheduler sinks the reads below the MFMAs that are to hide them
        __builtin_amdgcn_sched_barrier(0);
        compute(dd);
        BSG_TL_IF(2, t0 + d == 0);
        __builtin_amdgcn_sched_barrier(0);
      });
    }
  }
  BSG_TL_LOOP_END();

  // The channel halves meet in the ring (no load into it is in flight, no wave reads it any more).
  vmem_wait<0>();
  __syncthreads();
  // Each half finishes half of the row tiles: it hands the other half's to the other wave.
  constexpr int RH = RT / 2;
  static_for<RW>([&](auto rr) {
    if (rw != decltype(rr)::value) return;
    f32x4* const red = (f32x4*)ring_stage<PIECES, decltype(rr)::value>() + lane;
#pragma unroll
    for (int bi = 0; bi < RT; ++bi)
#pragma unroll
      for (int s = 0; s < NSUB; ++s)
        if (h == (bi < RH)) red[(bi * NSUB + s) * 64] = acc[bi][s];
  });
  __syncthreads();
  static_for<RW>([&](auto rr) {
    if (rw != decltype(rr)::value) return;
    const f32x4* const red = (const f32x4*)ring_stage<PIECES, decltype(rr)::value>() + lane;
#pragma unroll
    for (int bi = 0; bi < RT; ++bi)
#pragma unroll
      for (int s = 0; s < NSUB; ++s)
        if (h != (bi < RH) && s < nv)
          store_y<T, NSUB>(p, y0, st * 16, (rw * RT + bi) * NSUB + s, acc[bi][s] + red[(bi * NSUB + s) * 64]);
  });
  BSG_TL(4);
  BSG_TL_END(p, true);
}

// One form for every list source: beside these launches (15 us and more) the sort's code does not show.
#define BSG_R_FORM(...) \
  bsg_gemm_rows_kernel<_Float16, __VA_ARGS__, SEL_ANY_LIST>, bsg_gemm_rows_kernel<__bf16, __VA_ARGS__, SEL_ANY_LIST>
#define BSG_R(B, S, RW, D)                                                                       \
  {KIND_ROWS, 16 * B, S, 2 * RW, D, BSG_R_FORM(B, S, RW, D), BSG_R_FORM(B, S, RW, D), BSG_NO_2D_FORMS, \
   BSG_NO_SEL_FORMS}

}  // namespace
