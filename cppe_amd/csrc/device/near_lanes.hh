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
// Pair kernel of one apply against the staged form with chunks of 8 (same systems): FP32 0.156 -> 0.098 ms at
// 24,000 sites (chunks of 8), 0.468 -> 0.36 at 300,000 (chunks of 16); FP64 0.397 -> 0.235 and 1.45 -> 1.27 ms
// (chunks of 4: FP64 accumulators and the prefetched record leave room for more wavefronts then, and the
// undamped stages drop the exponential).
//
// POS: the type the positions are held in and subtracted in. double with R = float (untuned systems): displacements are
// formed in FP64 and rounded, and pairs are undamped from v >= 25 on, as in the thread-per-target form, so that an
// FP32 pair starts from no less than that form's. float: from offsets from the leaf's centre, each rounded, undamped
// from v >= 18 on. The former takes 0.128 ms at 24,000 sites and 0.52 at 300,000; its error of the field
// is 2.8e-7 there, 4.3e-7 with offsets and 8e-7 in the thread-per-target form (whose sums are one chain).

// Sums over the wavefront of every lane's f[t][c], formed in FP64; lane t receives those of target t. For FP32
// values 16 columns at a time go through LDS: four lanes add a column's 64 values (no slower than a tree of
// FP32 lane moves per value: 0.409 against 0.420 ms for the whole kernel at 300,000 sites).
constexpr int kSumCol = 65;  // 64 values and one of padding: no bank conflicts
template <int TS, int C>
__device__ __forceinline__ void target_sums(const float (&f)[TS][C], int, int lane, float* mem, double (&F)[C]) {
  constexpr int V = TS * C;
#pragma unroll
  for (int c = 0; c < C; ++c) F[c] = 0.0;
#pragma unroll
  for (int g = 0; g < V; g += 16) {
    wave_lds_barrier();
#pragma unroll
    for (int u = 0; u < 16; ++u)
      if (g + u < V) mem[u * kSumCol + lane] = f[(g + u) / C][(g + u) % C];
    wave_lds_barrier();
    const float* p = mem + (lane & 15) * kSumCol + (lane >> 4) * 16;
    double s       = 0.0;
#pragma unroll
    for (int r = 0; r < 16; ++r) s += (double)p[r];
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
#pragma unroll
    for (int c = 0; c < C; ++c) {  // column t C + c of target t, in lane (t C + c) - g
      const int v    = lane * C + c - g;
      const double x = __shfl(s, v & 15);
      if (v >= 0 && v < 16) F[c] = x;
    }
  }
}
template <int TS, int C>
__device__ __forceinline__ void target_sums(const double (&f)[TS][C], int T, int lane, float*, double (&F)[C]) {
#pragma unroll
  for (int c = 0; c < C; ++c) F[c] = 0.0;
#pragma unroll
  for (int t = 0; t < TS; ++t)
    if (t < T)
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const double v = wave_sum_f64(f[t][c]);
        if (lane == t) F[c] = v;
      }
}

// bytes of LDS per wavefront: the stage's skip bits, then (FP32) the columns of the sums
template <typename R>
constexpr int kLanesLds = sizeof(R) == 4 ? 16 * kSumCol * sizeof(float) : 64 * sizeof(int);

template <typename R, typename MU4>
struct LanesArgs {
  NearArgs a;
  SkipLists sk;
  const int4* items;
  int nitems;
  const long long* xoff;
  const int* xsrc;
  const long long *xspec, *xsplit;
  const MU4* mu4;
  const R* L;
  size_t lstride;
};

// A wavefront-uniform value the compiler knows nothing about from here on.
template <typename T>
__device__ __forceinline__ void opaque_scalar(T& v) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" : "+s"(v));
#endif
}

// The kernel's only argument, read from memory where it is called: what a kernel needs after its loops alone is
// then not held (and other scalars spilled) all through them.
template <typename T>
__device__ __forceinline__ const T& late_args(const T& now) {
#ifdef __HIP_DEVICE_COMPILE__
  auto p = __builtin_amdgcn_kernarg_segment_ptr();
  opaque_scalar(p);
  return *(const T*)(const void*)p;
#else
  return now;
#endif
}

template <int P, typename R, typename POS, bool DAMP, int MODE, typename MU4, bool WITH_L2P, int TS, bool B2, int K>
__global__ __launch_bounds__(256) void k_fmm_near_ls(LanesArgs<R, MU4> g) {
  using O        = Ops<KIND_M1, P, R>;
  const int lane = threadIdx.x & 63;
  const int w    = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
  if (w >= g.nitems) return;  // uniform per wavefront
  const NearArgs& a = g.a;
  extern __shared__ int lanes_lds[];
  int* const lds = lanes_lds + (threadIdx.x >> 6) * (kLanesLds<R> / (int)sizeof(int));
  const int4 it  = g.items[w];
  const int A   = __builtin_amdgcn_readfirstlane(it.x);
  const int i0  = __builtin_amdgcn_readfirstlane(it.y);
  const int T   = __builtin_amdgcn_readfirstlane(it.z);
  const int n   = a.n;
  const double cax = a.cx[A], cay = a.cy[A], caz = a.cz[A];
  const double4 pi = a.pos4[i0 + min(lane, T - 1)];  // lane t holds target t
  constexpr bool kAbs = sizeof(POS) == 8;
  // positions of the targets are scalars, and so are the damping rates where both fit the scalar registers; else a rate
  // is fetched from its lane at each pair, which the far stages, without damping, do not pay
  constexpr bool kRateScalar = TS * (3 * sizeof(POS) + sizeof(R)) <= 128;
  POS tx[TS], ty[TS], tz[TS];
  R td[kRateScalar ? TS : 1], f[TS][3 * K];
  const R vd = DAMP ? staged_di<R, B2>(a.damping, pi.w) : R(0);
  {
    const POS vx = (POS)(kAbs ? pi.x : pi.x - cax);
    const POS vy = (POS)(kAbs ? pi.y : pi.y - cay);
    const POS vz = (POS)(kAbs ? pi.z : pi.z - caz);
#pragma unroll
    for (int t = 0; t < TS; ++t) {
      tx[t] = read_lane(vx, t);
      ty[t] = read_lane(vy, t);
      tz[t] = read_lane(vz, t);
      if (kRateScalar) td[kRateScalar ? t : 0] = DAMP ? read_lane(vd, t) : R(0);
#pragma unroll
      for (int c = 0; c < 3 * K; ++c) f[t][c] = R(0);
    }
  }
  // the list, and positions in it as 32-bit numbers: the targets take most of the scalar registers, and the compiler
  // fetches each one that does not fit lane by lane in the pair loops
  const long long q0 = g.xoff[A];
  const int* src     = g.xsrc + q0;
  const int len      = (int)(g.xoff[A + 1] - q0);
  const int head     = min(len, ((int)(g.xspec[A] - q0) + 63) & ~63);  // (whole stages)
  const int near     = DAMP && g.xsplit ? (int)(g.xsplit[A] - q0) : len;
  constexpr POS kFar = POS(kAbs ? 1.0e8 : 1.0e4);  // lanes past the list: a source far away, no dipole
  double4 pn = make_double4(0.0, 0.0, 0.0, 0.0);
  MU4 mn[K];
  int jn = -1, jnn = 0;  // source of the record in pn, and of the stage after it
  auto gather = [&](int j) {
    jn = j;
    pn = a.pos4[j];
#pragma unroll
    for (int k = 0; k < K; ++k) mn[k] = g.mu4[(size_t)k * n + j];
  };
  if (lane < len) gather(src[lane]);
  if (lane < len - 64) jnn = src[64 + lane];
  // a loop for each form, not a branch per stage: with two forms of the pair in one loop the compiler keeps the
  // accumulators twice
  auto rate = [&](int t) { return !DAMP ? R(0) : kRateScalar ? td[kRateScalar ? t : 0] : read_lane(vd, t); };
  int q     = 0;
  auto walk = [&](auto far, int end, auto&& skips) {
    for (; q < end; q += 64) {
      StagedRec<R, K> r;
      POS sx = (POS)(kAbs ? pn.x : pn.x - cax);
      POS sy = (POS)(kAbs ? pn.y : pn.y - cay);
      POS sz = (POS)(kAbs ? pn.z : pn.z - caz);
      r.s    = (R)pn.w;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        r.m[3 * k]     = (R)mn[k].x;
        r.m[3 * k + 1] = (R)mn[k].y;
        r.m[3 * k + 2] = (R)mn[k].z;
      }
      const unsigned skip = skips(jn);
      if (lane >= len - q) {
        sx = sy = sz = kFar;
        r.s          = R(0);
#pragma unroll
        for (int c = 0; c < 3 * K; ++c) r.m[c] = R(0);
      }
      if (lane < len - q - 64) gather(jnn);                  // stage s + 1
      if (lane < len - q - 128) jnn = src[q + 128 + lane];  // stage s + 2: its source index
      int num = T;  // (anew in each stage: else the compiler compares once and keeps TS masks in scalar registers)
      opaque_scalar(num);
#pragma unroll
      for (int t = 0; t < TS; ++t)
        if (t < num)
          staged_pair<R, DAMP, B2, K, decltype(far)::value, false>((R)(tx[t] - sx), (R)(ty[t] - sy), (R)(tz[t] - sz),
                                                                   rate(t), r, f[t], keep_unless(skip, t));
    }
  };
  {  // the head: own sites stand at (site - start), partners in other leaves behind them
    const int ia = __builtin_amdgcn_readfirstlane(a.start[A]), na = __builtin_amdgcn_readfirstlane(a.count[A]);
    const ItemSkips its(g.sk, i0, T, lane, lds);
    const bool inside              = (unsigned)(its.site() - ia) < (unsigned)na;
    const unsigned long long other = __ballot(lane < its.n && !inside);
    walk(std::false_type{}, head, [&](int j) {
      const unsigned self = (unsigned)(j - i0) < (unsigned)T ? 1u << (j - i0) : 0u;
      return self | its.template run<true>(ia + q, inside) | its.template of<true>(j, other) | its.template rest<true>(j);
    });
  }
  const auto none = [](int) { return 0u; };
  walk(std::false_type{}, min(len, near), none);
  if (DAMP) walk(std::true_type{}, len, none);
  double F[3 * K];
  target_sums(f, T, lane, reinterpret_cast<float*>(lds), F);
  if (lane >= T) return;
  const auto& l     = late_args(g);
  const NearArgs& e = l.a;
  const int i      = i0 + lane;
  const double* ai = e.ainv;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    asm volatile("" ::: "memory");  // (one right-hand side's expansion in registers at a time)
    double* Fk = F + 3 * k;
    if constexpr (WITH_L2P) {
      R lx = R(0), ly = R(0), lz = R(0);
      O::l2p((R)(pi.x - e.cx[A]), (R)(pi.y - e.cy[A]), (R)(pi.z - e.cz[A]), &l.L[k * l.lstride + (size_t)A * O::LS], lx, ly, lz);
      Fk[0] += (double)lx;
      Fk[1] += (double)ly;
      Fk[2] += (double)lz;
    }
    const size_t o = 3 * (size_t)n * k;
    if (MODE == MODE_BAPPLY) {
      double a6[6];
#pragma unroll
      for (int c = 0; c < 6; ++c) a6[c] = ai[(size_t)c * n + i];
      const double m0 = e.src[o + i], m1 = e.src[o + n + i], m2 = e.src[o + 2 * (size_t)n + i];
      Fk[0] += a6[0] * m0 + a6[1] * m1 + a6[2] * m2;
      Fk[1] += a6[1] * m0 + a6[3] * m1 + a6[4] * m2;
      Fk[2] += a6[2] * m0 + a6[4] * m1 + a6[5] * m2;
    }
    e.out[o + i]                 = Fk[0];
    e.out[o + n + i]             = Fk[1];
    e.out[o + 2 * (size_t)n + i] = Fk[2];
  }
}
