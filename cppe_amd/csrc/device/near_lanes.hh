// Near field with lanes as sources (variants 7 and 8 of the B-apply near field).
//
// A work item is a chunk of at most TS targets of one leaf; the leaf's expanded near list is walked 64
// sources at a time, one per lane. A lane keeps its source (position, Thole scale, dipoles) in registers
// and the field of its sources at each of the chunk's targets (3 K accumulators a target); the targets'
// positions and damping rates are wavefront-uniform scalars. The pair loop therefore touches neither
// memory nor LDS -- in the form with lanes as (target, source slot) every pair reads its 32-byte FP32
// record from LDS, and the two 16-byte reads a wavefront needs per pair (a full wavefront's worth of LDS
// bandwidth each, shared by the CU's four SIMDs) take as long as the 20 vector instructions of an
// undamped pair. The lanes' fields are summed over the wavefront once per chunk.
// The records of the next stage and the source index of the one after are loaded while a stage is
// evaluated. Stages of the list's far class take the undamped pair (xsplit of the precision); excluded
// pairs and the targets themselves are skipped: both stand only in the head of the list (to xspec, the leaf's own sites
// first), whose stages look for them and have a loop of their own. Chunks of a leaf have equal sizes up to one, so that no
// short chunk walks the whole list for a few targets.
// Near field of one apply against the staged form with chunks of 8 (same systems; plus exclusions): FP32
// 0.156 -> 0.121 ms at 24,000 sites, 0.146 -> 0.123 at 60,000, 0.468 -> 0.388 at 300,000 (chunks of 16);
// FP64 0.397 -> 0.259, 0.56 -> 0.358, 1.45 -> 1.31 ms (chunks of 4: FP64 accumulators and the prefetched
// record leave room for more wavefronts then, and the undamped stages drop the exponential).
template <int P, typename R, bool DAMP, int MODE, typename MU4, bool WITH_L2P, int TS, bool B2, int K>
__global__ __launch_bounds__(256) void k_fmm_near_ls(NearArgs a, SkipLists sk, const int4* __restrict__ items,
                                                     int nitems,
                                                     const long long* __restrict__ xoff,
                                                     const int* __restrict__ xsrc,
                                                     const long long* __restrict__ xspec,
                                                     const long long* __restrict__ xsplit,
                                                     const MU4* __restrict__ mu4, const R* __restrict__ L,
                                                     size_t lstride) {
  using O        = Ops<KIND_M1, P, R>;
  const int lane = threadIdx.x & 63;
  const int w    = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
  if (w >= nitems) return;  // uniform per wavefront
  const int4 it = items[w];
  const int A   = __builtin_amdgcn_readfirstlane(it.x);
  const int i0  = __builtin_amdgcn_readfirstlane(it.y);
  const int T   = __builtin_amdgcn_readfirstlane(it.z);
  const int n   = a.n;
  const double cax = a.cx[A], cay = a.cy[A], caz = a.cz[A];
  const double4 pi = a.pos4[i0 + min(lane, T - 1)];  // lane t holds target t
  R tx[TS], ty[TS], tz[TS], td[TS], f[TS][3 * K];
  {
    const R vx = sizeof(R) == 8 ? (R)pi.x : (R)(pi.x - cax);
    const R vy = sizeof(R) == 8 ? (R)pi.y : (R)(pi.y - cay);
    const R vz = sizeof(R) == 8 ? (R)pi.z : (R)(pi.z - caz);
    const R vd = DAMP ? staged_di<R, B2>(a.damping, pi.w) : R(0);
#pragma unroll
    for (int t = 0; t < TS; ++t) {
      tx[t] = read_lane(vx, t);
      ty[t] = read_lane(vy, t);
      tz[t] = read_lane(vz, t);
      td[t] = DAMP ? read_lane(vd, t) : R(0);
#pragma unroll
      for (int c = 0; c < 3 * K; ++c) f[t][c] = R(0);
    }
  }
  const long long q0 = xoff[A], q1 = xoff[A + 1];
  const long long qs = min(q1, q0 + (xspec[A] - q0 + 63) / 64 * 64);  // stages of the head
  const long long qf = DAMP && xsplit ? xsplit[A] : q1;
  constexpr R kFar   = sizeof(R) == 4 ? R(1.0e4) : R(1.0e8);  // lanes past the list: a source far away, no dipole
  double4 pn = make_double4(0.0, 0.0, 0.0, 0.0);
  MU4 mn[K];
  int jn = -1, jnn = 0;  // source of the record in pn, and of the stage after it
  auto gather = [&](int j) {
    jn = j;
    pn = a.pos4[j];
#pragma unroll
    for (int k = 0; k < K; ++k) mn[k] = mu4[(size_t)k * n + j];
  };
  if (lane < q1 - q0) gather(xsrc[q0 + lane]);
  if (lane < q1 - q0 - 64) jnn = xsrc[q0 + 64 + lane];
  // a loop for each form, not a branch per stage: with two forms of the pair in one loop the compiler keeps the
  // accumulators twice
  long long q = q0;
  auto walk   = [&](auto far, long long end, auto&& skips) {
    for (; q < end; q += 64) {
      StagedRec<R, K> r;
      r.x = sizeof(R) == 8 ? (R)pn.x : (R)(pn.x - cax);
      r.y = sizeof(R) == 8 ? (R)pn.y : (R)(pn.y - cay);
      r.z = sizeof(R) == 8 ? (R)pn.z : (R)(pn.z - caz);
      r.s = (R)pn.w;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        r.m[3 * k]     = (R)mn[k].x;
        r.m[3 * k + 1] = (R)mn[k].y;
        r.m[3 * k + 2] = (R)mn[k].z;
      }
      const unsigned skip = skips(jn);
      if (q1 - q < 64 && lane >= q1 - q) {
        r.x = r.y = r.z = kFar;
        r.s = R(0);
#pragma unroll
        for (int c = 0; c < 3 * K; ++c) r.m[c] = R(0);
      }
      if (lane < q1 - q - 64) gather(jnn);                   // stage s + 1
      if (lane < q1 - q - 128) jnn = xsrc[q + 128 + lane];  // stage s + 2: its source index
#pragma unroll
      for (int t = 0; t < TS; ++t)
        if (t < T)
          staged_pair<R, DAMP, B2, K, decltype(far)::value, false>(tx[t] - r.x, ty[t] - r.y, tz[t] - r.z, td[t], r, f[t],
                                                                   skip >> t & 1u);
    }
  };
  {  // the head: own sites stand at q0 + (site - start), partners in other leaves behind them
    const int ia = __builtin_amdgcn_readfirstlane(a.start[A]), na = __builtin_amdgcn_readfirstlane(a.count[A]);
    __shared__ int2 mem[4][64];
    unsigned ent;
    const ItemSkips its(sk, i0, T, lane, mem[threadIdx.x >> 6], ent);
    const int at                   = (int)(ent & kSkipSite) - ia;
    const bool inside              = lane < its.n && (unsigned)at < (unsigned)na;
    const unsigned long long other = __ballot(lane < its.n && !inside);
    walk(std::false_type{}, qs, [&](int j) {
      const int qr               = (int)(q - q0);
      const unsigned long long m = other | __ballot(inside && (unsigned)(at - qr) < 64u);
      unsigned s                 = (unsigned)(j - i0) < (unsigned)T ? 1u << (j - i0) : 0u;
      if (m != 0 || its.n > 64) s |= its.template of<true>(j, m);
      return s;
    });
  }
  const auto none = [](int) { return 0u; };
  walk(std::false_type{}, min(q1, qf), none);
  if (DAMP) walk(std::true_type{}, q1, none);
  double F[3 * K];
#pragma unroll
  for (int c = 0; c < 3 * K; ++c) F[c] = 0.0;
#pragma unroll
  for (int t = 0; t < TS; ++t)
    if (t < T)
#pragma unroll
      for (int c = 0; c < 3 * K; ++c) {
        const double v = (double)sym_wave_sum(f[t][c]);
        if (lane == t) F[c] = v;
      }
  if (lane >= T) return;
  const int i      = i0 + lane;
  const double* ai = a.ainv;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    double* Fk = F + 3 * k;
    if constexpr (WITH_L2P) {
      R lx = R(0), ly = R(0), lz = R(0);
      O::l2p((R)(pi.x - cax), (R)(pi.y - cay), (R)(pi.z - caz), &L[k * lstride + (size_t)A * O::LS], lx, ly, lz);
      Fk[0] += (double)lx;
      Fk[1] += (double)ly;
      Fk[2] += (double)lz;
    } else {
      (void)L;
      (void)lstride;
    }
    const size_t o = 3 * (size_t)n * k;
    if (MODE == MODE_BAPPLY) {
      double a6[6];
#pragma unroll
      for (int c = 0; c < 6; ++c) a6[c] = ai[(size_t)c * n + i];
      const double m0 = a.src[o + i], m1 = a.src[o + n + i], m2 = a.src[o + 2 * (size_t)n + i];
      Fk[0] += a6[0] * m0 + a6[1] * m1 + a6[2] * m2;
      Fk[1] += a6[1] * m0 + a6[3] * m1 + a6[4] * m2;
      Fk[2] += a6[2] * m0 + a6[4] * m1 + a6[5] * m2;
    }
    a.out[o + i]                 = Fk[0];
    a.out[o + n + i]             = Fk[1];
    a.out[o + 2 * (size_t)n + i] = Fk[2];
  }
}
