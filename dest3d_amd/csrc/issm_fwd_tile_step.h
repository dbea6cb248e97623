// One step of k_local_tile (issm_fwd_tile.hip): 64 state columns, 16 of them the wave's.  Included where it runs, inside a loop
// over n0 and with DEEP defined: the usual form (false), which, where some tile of the wave's columns is out of range (bf16 inputs), breaks
// off with nothing stored (ANY) or ends the loop with the step, and, ANY only, the form that has no range (true).  (Text and not a function: as an inlined lambda
// the usual form is allocated differently, fp32 1 to 4 % slower.)
    const int bad_seen = IOB && !ANY ? __hip_atomic_load(&s.bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : 0;
    const float A2[4] = {rA.x * LOG2E, rA.y * LOG2E, rA.z * LOG2E, rA.w * LOG2E};
    float bias[4] = {rbias.x * bias_on, rbias.y * bias_on, rbias.z * bias_on, rbias.w * bias_on};
#pragma unroll
    for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(bias[r]));   // (multiplied and added at once, every sum would begin as a copy of its dt)
    // the lane's columns this step: c .. c + 3, of which the first `skip` are not its own
    const int c = EDGE ? min(n0 + ncol, p.N - 4) : n0 + ncol, skip = EDGE ? n0 + ncol - c : 0;
    auto put = [&](float* q, f4 v) {   // q: where column c goes
      if constexpr (!EDGE) {
        *(f4*)q = v;
      } else if (skip == 0) {
        st_f4_any(q, v);
      } else {
#pragma unroll
        for (int j = 1; j < 4; ++j)
          if (j >= skip) q[j] = v[j];
      }
    };
    // the next step, whose operands are requested once this one's have been used (the last one asks for its own once more: no branch)
    const int nn = EDGE ? (n0 + NS < p.N ? n0 + NS : n0) : min(n0 + NS, p.N - NS);

    // ---- dt transform and the running sums of the tiles
    float dtp[16], dummy[16];
    {
      float pre[16];
      hand_over(rdt, pre);
#pragma unroll
      for (int k = 0; k < 16; ++k) pre[k] += bias[k & 3];
      ISSM_REQUEST_DT(nn)
      dt_transform<false, 16>(p, pre, dtp, dummy);
      if constexpr (EDGE) {
        if (nvalid < CS || n0 + NS > p.N) {  // uniform
#pragma unroll
          for (int k = 0; k < 16; ++k)
            if (16 * (k >> 2) + i >= nvalid || (k & 3) < skip) dtp[k] = 0.0f;
        }
      }
    }
    float pc[16], up[16], et[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) pc[k] = dtp[k] * A2[k & 3];
    row_scans(pc);
#pragma unroll
    for (int k = 0; k < 16; ++k) up[k] = ex2(pc[k]);
#pragma unroll
    for (int k = 0; k < 16; ++k) et[k] = row_lane<15>(up[k]);  // whole-tile decay of the lane's columns
    if (!DEEP) {
#pragma unroll
      for (int k = 0; k < 16; k += 2) etmin = fminf(etmin, fminf(et[k], et[k + 1]));
    }
    if constexpr (IOB && !DEEP) {
      const bool out = __ballot(!(etmin >= thr)) != 0ull;   // wave-uniform; no barrier in the loop
      if constexpr (ANY) {
        if (out) break;
      } else {
        if (out) s.bad = 1;
        stop = out | (__builtin_amdgcn_readfirstlane(bad_seen) != 0);
      }
    }
    {  // the chunk's total decay (natural logarithm), four adjacent columns per lane group.  All 16 lanes of a group
       // store the same values to the same place: a store under a lane condition sits behind a branch, and the waits
       // for the requests in flight -- counted in order with the stores -- would then have to assume it away and wait
       // for every store as well.
      f4 tot;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        tot[r] = row_lane<15>((((pc[r] + pc[4 + r]) + pc[8 + r]) + pc[12 + r]) * LN2);
      }
      put(cdst + c, tot);
    }

    // ---- operands
    float bv[16], cv[16], w16[EDGE || DEEP ? 16 : 1];
    hand_over(rC, cv);
    ISSM_REQUEST_C(nn)
    if constexpr (EDGE) {
      if (nvalid < CS) {  // uniform
#pragma unroll
        for (int k = 0; k < 16; ++k)
          if (16 * (k >> 2) + i >= nvalid) cv[k] = 0.0f;   // (rows of M past the end come out as zero)
      }
    }
    hand_over(rB, bv);
    ISSM_REQUEST_B(nn)
    if constexpr (DEEP) {
#pragma unroll
      for (int J = 0; J < 4; ++J) {
#pragma unroll
        for (int k = 4 * J; k < 4 * J + 4; ++k) w16[k] = dtp[k] * bv[k];
        far_diagonal(cv + 4 * J, w16 + 4 * J, pc + 4 * J, macc[J]);
#pragma unroll
        for (int k = 4 * J; k < 4 * J + 4; ++k) cv[k] *= up[k];
      }
    } else if constexpr (EDGE) {
      // diagonal blocks, before anything else needs registers: W takes the place of B and dt', C up that of C.  fp32 matrix
      // instructions: k-slot kg of instruction r <-> the lane's column r; the blocks' chains are interleaved.
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        w16[k] = dtp[k] * bv[k] * ex2(-pc[k]);
        cv[k] *= up[k];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int J = 0; J < 4; ++J) macc[J] = mfma4(cv[4 * J + r], w16[4 * J + r], macc[J]);
    }
    auto cu = [&](int k) { return EDGE || DEEP ? cv[k] : cv[k] * up[k]; };
    Fr U[4];
#pragma unroll
    for (int J = 0; J < 4; ++J) U[J] = make_frag<SPLIT>(cu(4 * J), cu(4 * J + 1), cu(4 * J + 2), cu(4 * J + 3));
    f4 sacc[PT];
#pragma unroll
    for (int pt = 0; pt < PT; ++pt) sacc[pt] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int J = 0; J < 4; ++J) {
      float W[4], V[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = 4 * J + r;
        if constexpr (EDGE || DEEP) W[r] = w16[k];
        else W[r] = dtp[k] * bv[k] * ex2(-pc[k]);
        V[r] = W[r] * (DEEP ? ex2(row_lane<15>(pc[k]) - pc[k]) : et[k]);
      }
      if constexpr (!EDGE && !DEEP) {
        const Fr f = make_frag<SPLIT>(W[0], W[1], W[2], W[3]);
        macc[J] = frag_product<SPLIT>(U[J], f, macc[J]);
      }
      // V serves the block below the diagonal one (J < 3) and the chunk state: always as a (hi, lo) pair
      const Frag<true> fv = make_frag<true>(V[0], V[1], V[2], V[3]);
      if (J < 3) {
        Fr f;
        f.h = fv.h;
        f.l = fv.l;
        macc[4 + J] = frag_product<SPLIT>(U[J + 1], f, macc[4 + J]);
      }
      if (J < 2) {
        float V2[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) V2[r] = V[r] * et[4 * (J + 1) + r];
        const Fr f = make_frag<SPLIT>(V2[0], V2[1], V2[2], V2[3]);
        macc[7 + J] = frag_product<SPLIT>(U[J + 2], f, macc[7 + J]);
        if (J == 0) {
          const Fr g = make_frag<SPLIT>(V2[0] * et[8], V2[1] * et[9], V2[2] * et[10], V2[3] * et[11]);
          macc[9] = frag_product<SPLIT>(U[3], g, macc[9]);
        }
      }
      // chunk state: what the earlier tiles have summed decays across tile J (accumulator r <-> the lane's column r),
      // then V of tile J, lane and register roles exchanged, meets x^T of tile J's rows
      {
        if (J > 0) {
#pragma unroll
          for (int pt = 0; pt < PT; ++pt)
#pragma unroll
            for (int r = 0; r < 4; ++r) sacc[pt][r] *= et[4 * J + r];
        }
        // (wider head dimensions: keep the scheduler from fetching every tile's x fragments ahead of time, which
        // costs more registers than there are)
        if (PT > 2 || DEEP) __builtin_amdgcn_sched_barrier(0);
        const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        const bf4 th = exact_bf4(mfma_bf16k(fv.h, ident, zero)), tlo = exact_bf4(mfma_bf16k(fv.l, ident, zero));
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) {
          const int xo = (16 * pt + i) * LDT + 16 * J + 4 * kg;
          const bf4 xh = *(const bf4*)(s.xt_hi + xo);
          sacc[pt] = mfma_bf16k(tlo, xh, sacc[pt]);
          if (SPLIT) {
            const bf4 xl = *(const bf4*)(s.xt_lo + xo);
            sacc[pt] = mfma_bf16k(th, xl, sacc[pt]);
          }
          sacc[pt] = mfma_bf16k(th, xh, sacc[pt]);
        }
      }
    }
    // S^T block: lane (p = i, kg) holds columns n0 + ncol .. + 3 of state row 16 pt + i
    if (FULLP) {  // every state row exists: plain stores (see the note at the chunk's total decay)
#pragma unroll
      for (int pt = 0; pt < PT; ++pt) put(sdst + (16 * pt + i) * p.N + c, sacc[pt]);
    } else if constexpr (!EDGE) {   // (rows past the last lie behind the slab's end, where a store is dropped: no branch either)
#pragma unroll
      for (int pt = 0; pt < PT; ++pt)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, sacc[pt]), slab, (unsigned)((16 * pt + i) * p.N + c) * 4u, 0, 0);
    } else {
#pragma unroll
      for (int pt = 0; pt < PT; ++pt)
        if (16 * pt + i < p.P) put(sdst + (16 * pt + i) * p.N + c, sacc[pt]);
    }
