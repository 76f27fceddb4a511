// Host-side launchers of the fused kernels: the pass-shape registries
// (instantiated per transform length in ns2d_pass_tu.hip), the row/column pass
// launches, the real-field forward transform and the measures reduction.
#include "ns2d_kernels.hpp"

namespace ns2d {
// ---------------------------------------------------------------------------
// host-side launchers (template dispatch on the transform lengths)
// ---------------------------------------------------------------------------

// the shape instantiations, one function per translation unit of
// ns2d_pass_tu.hip (built once per length range, ascending)
#define NS2D_PASS_TUS(X) X(8, 128) X(256, 256) X(512, 512) X(1024, 1024) X(2048, 2048) X(4096, 4096)
#define NS2D_TU_DECL(LO, HI)                           \
  void kv_add_##LO##_##HI(std::vector<KVariant>& v); \
  void rv_add_##LO##_##HI(std::vector<RVariant>& v);
NS2D_PASS_TUS(NS2D_TU_DECL)
#undef NS2D_TU_DECL

const std::vector<KVariant>& kvariant_table() {
  static const std::vector<KVariant> t = [] {
    std::vector<KVariant> v;
#define NS2D_TU_CALL(LO, HI) kv_add_##LO##_##HI(v);
    NS2D_PASS_TUS(NS2D_TU_CALL)
#undef NS2D_TU_CALL
    return v;
  }();
  return t;
}

// FNV-1a hash of the compiled column-pass shapes of length nx and row-pass
// shapes of length ny (a tuned schedule names shapes by index, valid only for
// the same tables)
unsigned long long shape_table_hash(int nx, int ny) {
  unsigned long long h = 1469598103934665603ull;
  auto mix = [&](int x) {
    for (int b = 0; b < 4; ++b) {
      h ^= (unsigned long long)((x >> (8 * b)) & 0xff);
      h *= 1099511628211ull;
    }
  };
  for (const KVariant& v : kvariant_table())
    if (v.L == nx) {
      const int f[] = {v.L, v.C, v.T, v.KS, v.PS, v.OFF, v.PK, v.W, v.PF};
      for (int x : f) mix(x);
    }
  mix(-1);
  for (const RVariant& v : rvariant_table())
    if (v.NY == ny) {
      const int f[] = {v.NY, v.TLR, v.PAIRS, v.W, v.PFR};
      for (int x : f) mix(x);
    }
  return h;
}

const std::vector<RVariant>& rvariant_table() {
  static const std::vector<RVariant> t = [] {
    std::vector<RVariant> v;
#define NS2D_TU_CALL(LO, HI) rv_add_##LO##_##HI(v);
    NS2D_PASS_TUS(NS2D_TU_CALL)
#undef NS2D_TU_CALL
    return v;
  }();
  return t;
}

static const KVariant* find_kvariant(int nx, int idx) {
  int n = 0;
  for (const KVariant& v : kvariant_table()) {
    if (v.L != nx) continue;
    if (n++ == idx) return &v;
  }
  return nullptr;
}

// Every member of the batch must run a pass with inverse transforms (KS as
// compiled) and share nyf and nyc.
hipError_t launch_kpass_batched(int nx, int nyc, int band, int variant, const KPassArgs* tab, int members, hipStream_t s) {
  const KVariant* v = find_kvariant(nx, variant);
  if (!v || !v->batched[band ? 1 : 0]) return hipErrorInvalidValue;
  const int per = v->groups(nyc) * v->KS;
  hipLaunchKernelGGL(v->batched[band ? 1 : 0], dim3(per * members), dim3(v->T), 0, s, tab, per);
  return hipGetLastError();
}

static int k_index(int L, int C, int T, int KS, int PS, int OFF, int PF) {
  int n = 0;
  for (const KVariant& v : kvariant_table()) {
    if (v.L != L) continue;
    if (v.C == C && v.T == T && v.KS == KS && v.PS == PS && v.OFF == OFF && v.PF == PF && v.PK == 0 && v.W == 1) return n;
    ++n;
  }
  return 0;
}

static int r_index(int NY, int TLR, int PAIRS, int PFR) {
  int n = 0;
  for (const RVariant& v : rvariant_table()) {
    if (v.NY != NY) continue;
    if (v.TLR == TLR && v.PAIRS == PAIRS && v.PFR == PFR) return n;
    ++n;
  }
  return 0;
}

// Default column-pass shape for passes over nyc columns: index 0 of its length
// (at 4096 the unpacked 1024-thread shape with the 16-slot padding: 320.5
// against 326.9 us per RK4CN launch for the 512-thread one, 444.2 against
// 445.0 us for CN-AB4's heavier epilogue, in alternating bench runs) where
// the columns roughly fill the CUs once; with many more columns, shapes that
// redo less of the forward transform, with fewer, shapes of one column per
// workgroup.  Column pass, us per launch, against index 0:
//   128   > 512 columns   2 columns, 4 points per lane  (128x4096 RK4CN step 140 / 151)
//   256   > 1024          2 splits instead of 4         2049 columns 21.7 / 26.5
//   512   > 400           2 columns, 2 splits           513: 21.2 / 22.0, 2049: 37.5 / 53.2
//   512   <= 400          index 0 on two line buffers   257: 15.1 / 15.7
//   1024  <= 512          index 0 on two line buffers   341: 22.6 / 23.6 (513: 28.1 / 24.3)
//   1024  > 700           2 columns of 512 threads      1025: 41.7 / 45.6, 2049: 76.7 / 97.3
//   2048  <= 300          1 column, 2 splits            257: 27.5 / 34.0
//   2048  <= 700          1 column                      513: 40.8 / 46.0, 683: 45.7 / 46.7
//   4096  301 .. 700      1 column, exchanges of doubles 513: 96.2 / 104.3 (257: 54.8 / 49.9)
int kpass_default_variant(int nx, int nyc) {
  if (nx == 128 && nyc > 512) return k_index(128, 2, 64, 4, 3, 1, 0);
  if (nx == 256 && nyc > 1024) return k_index(256, 1, 64, 2, 3, 1, 0);
  if (nx == 512) return nyc > 400 ? k_index(512, 2, 256, 2, 4, 8, 0) : k_index(512, 1, 128, 4, 3, 1, 4);
  if (nx == 1024 && nyc <= 512) return k_index(1024, 1, 256, 2, 4, 1, 4);
  if (nx == 1024 && nyc > 700) return k_index(1024, 2, 512, 2, 4, 8, 0);
  if (nx == 2048 && nyc <= 300) return k_index(2048, 1, 256, 2, 3, 1, 0);
  if (nx == 2048 && nyc <= 700) return k_index(2048, 1, 256, 1, 3, 1, 0);
  if (nx == 4096 && nyc > 300 && nyc <= 700) return k_index(4096, 1, 512, 1, 3, 1, 2);
  return 0;
}

// Default row-pass shape.  Below 2048 rows a launch is one chain of latencies:
// up to 1024 points a single row on two teams (rpass_team_body).  From 2048 rows
// on the pass is bound by its traffic:
//   up to 512   row pairs in whole waves (2048x512 171.6 us per step against 174.0 on
//               teams, 4096x512 294 / 305, 4096x64 212 / 254)
//   1024        single rows, the fields loaded as needed: two waves per SIMD
//               (2048x1024 263.5 / 264.8, 4096 rows 44.4 / 51.5 us per launch)
// CN-AB4 forms max|w| in every step, which row pairs do with one transform for two
// rows: 1024 points from 1024 rows on 43.9 us per step against 48.4 (1024^2),
// 81.3 / 88.1 (2048x1024).  4096: index 0, exchanges of doubles; up to 512 rows the
// 512-thread shape (22.6 / 23.3 us per launch); with CN-AB4 the fields loaded as
// needed (443.8 against 463 us per step).
int rpass_default_variant(int nx, int ny, bool ab4) {
  const bool tall = nx >= 2048;
  switch (ny) {
    case 8: return tall ? 0 : r_index(8, 4, 1, 3);
    case 16: return tall ? 0 : r_index(16, 8, 1, 3);
    case 32: return tall ? 0 : r_index(32, 16, 1, 6);
    case 64: return tall ? 0 : r_index(64, 16, 1, 14);
    case 128: return tall ? 0 : r_index(128, 64, 1, 14);
    case 256: return tall ? r_index(256, 32, 2, 0) : r_index(256, 64, 1, 6);
    case 512: return tall ? r_index(512, 64, 4, 0) : r_index(512, 64, 1, 6);
    case 1024:
      if (ab4 && nx >= 1024) return r_index(1024, 256, 1, 1);
      return tall ? r_index(1024, 64, 1, 2) : r_index(1024, 64, 1, 6);
    case 4096:
      if (nx <= 512) return r_index(4096, 512, 1, 2);
      return ab4 ? r_index(4096, 256, 1, 18) : 0;
    default: return 0;
  }
}

int kpass_variant_count(int nx) {
  int n = 0;
  for (const KVariant& v : kvariant_table()) n += v.L == nx;
  return n;
}

int kpass_variant_info(int nx, int idx, int* C, int* E, int* T, int* KS) {
  const KVariant* v = find_kvariant(nx, idx);
  if (!v) return -1;
  *C = v->C;
  *E = v->L * v->C / v->T;
  *T = v->T;
  *KS = v->KS;
  return 0;
}

int kpass_variant_extra(int nx, int idx, int* W, int* PS, int* OFF, int* PK) {
  const KVariant* v = find_kvariant(nx, idx);
  if (!v) return -1;
  *W = v->W;
  *PS = v->PS;
  *OFF = v->OFF;
  *PK = (v->PK != 0) | ((v->PF & 1) << 1) | ((v->PK == 2) << 2) | (((v->PF & 2) != 0) << 6) |
        (((v->PF & 4) != 0) << 7) | (((v->PF & 8) != 0) << 5);
  return 0;
}

bool kpass_has_band(int nx, int variant) {
  const KVariant* v = find_kvariant(nx, variant);
  return v && v->kern[1];
}

// Launch the kpass for an nx-point column transform.  A pass without inverse
// transforms (an RHS evaluation) runs one workgroup per column group: split
// workgroups exist only to share the inverse fields.
hipError_t launch_kpass(int nx, int variant, const KPassArgs& a, hipStream_t s) {
  const KVariant* v = find_kvariant(nx, variant);
  if (!v || !v->kern[a.band ? 1 : 0]) return hipErrorInvalidValue;
  const int groups = v->groups(a.nyc);
  const int splits = (a.mode & KP_INV) ? v->KS : 1;
  // A last column group holding a single column (unpacked, KS = 1, more than
  // one column per group) runs as two half items: it would otherwise be the
  // one workgroup left when every CU has finished its share
  KPassArgs b = a;
  b.last_split = (v->KS == 1 && v->PK == 0 && v->C > 1 && (a.mode & KP_INV) && a.nyc % v->C == 1) ? 1 : 0;
  hipLaunchKernelGGL(v->kern[a.band ? 1 : 0], dim3(groups * splits + b.last_split), dim3(v->T), 0, s, b);
  return hipGetLastError();
}

static const RVariant* find_rvariant(int ny, int idx) {
  int n = 0;
  for (const RVariant& v : rvariant_table()) {
    if (v.NY != ny) continue;
    if (n++ == idx) return &v;
  }
  return nullptr;
}

hipError_t launch_rpass_batched(int nx, int ny, int band, int variant, const RPassArgs* tab, int members, hipStream_t s) {
  const RVariant* v = find_rvariant(ny, variant);
  if (!v) return hipErrorInvalidValue;
  const int units = (v->PFR & 7) >= 2 ? nx : nx / 2;   // rows or row pairs
  const int per = (units + v->PAIRS - 1) / v->PAIRS;
  hipLaunchKernelGGL(v->batched[band ? 1 : 0], dim3(per * members), dim3(v->TLR * v->PAIRS * rpass_teams(v->PFR)), 0, s, tab,
                     per);
  return hipGetLastError();
}

int rpass_variant_count(int ny) {
  int n = 0;
  for (const RVariant& v : rvariant_table()) n += v.NY == ny;
  return n;
}

int rpass_variant_info(int ny, int idx, int* TLR, int* E, int* T, int* PAIRS) {
  const RVariant* v = find_rvariant(ny, idx);
  if (!v) return -1;
  *TLR = v->TLR;
  *E = v->NY / v->TLR;
  *T = v->TLR * v->PAIRS;
  *PAIRS = v->PAIRS;
  return 0;
}

int rpass_variant_extra(int ny, int idx, int* W, int* PS, int* OFF, int* PK) {
  const RVariant* v = find_rvariant(ny, idx);
  if (!v) return -1;
  *W = v->W;
  *PS = 3;
  *OFF = 1;
  const int pm = v->PFR & 7;
  *PK = ((pm == 1 || pm == 3 || pm == 4) << 1) | ((pm >= 2) << 3) | ((pm == 4 || pm == 5 || pm == 7) << 4) | ((pm >= 6) << 8) | (((v->PFR & 8) != 0) << 5) |
        (((v->PFR & 16) != 0) << 6);
  return 0;
}

hipError_t launch_rpass(int nx, int ny, int variant, const RPassArgs& a, hipStream_t s) {
  const RVariant* v = find_rvariant(ny, variant);
  if (!v) return hipErrorInvalidValue;
  const int units = (v->PFR & 7) >= 2 ? nx : nx / 2;   // rows or row pairs
  const int b = a.band ? 1 : 0;
  hipLaunchKernelGGL((a.mode & RP_CFL) ? v->cfl[b] : v->kern[b], dim3((units + v->PAIRS - 1) / v->PAIRS),
                     dim3(v->TLR * v->PAIRS * rpass_teams(v->PFR)), 0, s, a);
  return hipGetLastError();
}

template <int NY>
struct R2CCfg {
  static constexpr int T = NY >= 1024 ? 256 : (NY / 4 < 64 ? 64 : NY / 4);
};

template <int NY>
static hipError_t launch_r2c_rows_t(int nx, const double* in, double2* out, const double2* tw, int ld,
                                    hipStream_t s) {
  constexpr int T = R2CCfg<NY>::T;
  hipLaunchKernelGGL((r2c_rows_kernel<NY, T>), dim3(nx), dim3(T), 0, s, in, out, tw, ld);
  return hipGetLastError();
}

hipError_t launch_r2c_rows(int nx, int ny, const double* in, double2* out, const double2* tw, int ld,
                           hipStream_t s) {
  switch (ny) {
    case 8: return launch_r2c_rows_t<8>(nx, in, out, tw, ld, s);
    case 16: return launch_r2c_rows_t<16>(nx, in, out, tw, ld, s);
    case 32: return launch_r2c_rows_t<32>(nx, in, out, tw, ld, s);
    case 64: return launch_r2c_rows_t<64>(nx, in, out, tw, ld, s);
    case 128: return launch_r2c_rows_t<128>(nx, in, out, tw, ld, s);
    case 256: return launch_r2c_rows_t<256>(nx, in, out, tw, ld, s);
    case 512: return launch_r2c_rows_t<512>(nx, in, out, tw, ld, s);
    case 1024: return launch_r2c_rows_t<1024>(nx, in, out, tw, ld, s);
    case 2048: return launch_r2c_rows_t<2048>(nx, in, out, tw, ld, s);
    case 4096: return launch_r2c_rows_t<4096>(nx, in, out, tw, ld, s);
    default: return hipErrorInvalidValue;
  }
}

// Between the host layout [Nx][nyf] (contiguous rows, what callers pass) and
// the device k-space layout (kidx, padding columns ky >= nyf zero): dir 0 packs
// src (host layout) into dst, dir 1 unpacks src into dst (host layout).
// kc2 > 0: modes with |k|^2 >= kc2 lie outside the 2/3 filter's disk.  dir 0:
// *spill = epoch when one of them is not zero (NaN counts as not zero); dir 1:
// they are zero and not read (NaN once the state has blown up: a NaN in any
// mode has then reached every mode of the disk, and 0 * NaN is what the
// filter leaves).
// A transpose for the column-major layout: 32 x 32 tiles through LDS (rows one
// 16-B slot longer than the tile, so that a column's reads fall on distinct
// banks), both sides in runs of 512 B.  Bound by memory: 2 x 16 B per mode.
constexpr int RELAYOUT_TILE = 32;
__global__ __launch_bounds__(256) void relayout_kernel(const double2* __restrict__ src, double2* __restrict__ dst,
                                                       int nyf, int ld, int nx, int dir, long kc2,
                                                       unsigned long long* __restrict__ spill,
                                                       unsigned long long epoch) {
  constexpr int RT = RELAYOUT_TILE, ROWS = 256 / RT;
  __shared__ double2 tile[RT][RT + 1];   // [x][ky]
  const int x0 = (int)blockIdx.y * RT, k0 = (int)blockIdx.x * RT;
  const int tx = (int)threadIdx.x % RT, ty = (int)threadIdx.x / RT;
  auto outside = [&](int x, int ky) -> bool {
    const long kx = kx_of_row(x, nx);
    return kc2 > 0 && kx * kx + (long)ky * ky >= kc2;
  };
  if (dir == 0) {
    bool spills = false;
#pragma unroll
    for (int r = ty; r < RT; r += ROWS) {
      const int x = x0 + r, ky = k0 + tx;
      const bool in = x < nx && ky < nyf;
      const double2 v = in ? src[(size_t)x * nyf + ky] : make_double2(0.0, 0.0);
      spills = spills || (in && outside(x, ky) && !(v.x == 0.0 && v.y == 0.0));
      tile[r][tx] = v;
    }
    if (spills) *spill = epoch;
    __syncthreads();
#pragma unroll
    for (int r = ty; r < RT; r += ROWS) {
      const int x = x0 + tx, ky = k0 + r;
      if (x < nx && ky < ld) dst[kidx(x, ky, ld, nx)] = tile[tx][r];
    }
  } else {
    const double2 z = cscale(0.0, src[kidx(1, 0, ld, nx)]);
#pragma unroll
    for (int r = ty; r < RT; r += ROWS) {
      const int x = x0 + tx, ky = k0 + r;
      if (x < nx && ky < nyf) tile[tx][r] = outside(x, ky) ? z : src[kidx(x, ky, ld, nx)];
    }
    __syncthreads();
#pragma unroll
    for (int r = ty; r < RT; r += ROWS) {
      const int x = x0 + r, ky = k0 + tx;
      if (x < nx && ky < nyf) dst[(size_t)x * nyf + ky] = tile[r][tx];
    }
  }
}

hipError_t launch_relayout(const double2* src, double2* dst, int nx, int nyf, int ld, int dir, long kc2,
                           unsigned long long* spill, unsigned long long epoch, hipStream_t s) {
  constexpr int RT = RELAYOUT_TILE;
  hipLaunchKernelGGL(relayout_kernel, dim3((ld + RT - 1) / RT, (nx + RT - 1) / RT), dim3(256), 0, s, src, dst, nyf, ld, nx, dir, kc2, spill, epoch);
  return hipGetLastError();
}

// The host used to read a handle's status words, change them and write them
// back, two copies and two waits per call; as launches on the handle's stream
// they leave one copy and one wait (64x64, ten steps from a new state: 467 -> 439 us).
__device__ __forceinline__ bool stat_check(unsigned long long* st) {
  const unsigned long long m = st[STAT_WMAX_CUR];
  // a NaN maximum also counts (the reference's >= test would let it pass)
  if (!(__longlong_as_double((long long)m) < MAX_VORT_LIM) && st[STAT_FIRST_BAD] == ~0ull)
    st[STAT_FIRST_BAD] = st[STAT_ITER];
  st[STAT_WMAX_LAST] = m;
  st[STAT_WMAX_CUR] = 0ull;
  return st[STAT_FIRST_BAD] == ~0ull;
}

__global__ __launch_bounds__(64) void stat_kernel(unsigned long long* st, int op) {
  if (threadIdx.x != 0) return;
  switch (op) {
    case STAT_OP_RESET:
      st[STAT_WMAX_CUR] = st[STAT_WMAX_LAST] = st[STAT_ITER] = st[STAT_CFL] = 0ull;
      st[STAT_FIRST_BAD] = ~0ull;
      break;
    case STAT_OP_CHECK: (void)stat_check(st); break;
    case STAT_OP_CLEAR_WMAX: st[STAT_WMAX_CUR] = 0ull; break;
    default: st[STAT_CFL] = 0ull; break;
  }
}

__global__ __launch_bounds__(64) void stat_check_all_kernel(unsigned long long* const* stats, int n, int* bad) {
  __shared__ int first[64];
  const int tid = (int)threadIdx.x;
  int f = n;
  for (int i = tid; i < n; i += 64)
    if (!stat_check(stats[i]) && i < f) f = i;
  first[tid] = f;
  __syncthreads();
  if (tid == 0) {
    for (int t = 1; t < 64; ++t) f = first[t] < f ? first[t] : f;
    *bad = f < n ? f : -1;
  }
}

hipError_t launch_stat(unsigned long long* stat, int op, hipStream_t s) {
  hipLaunchKernelGGL(stat_kernel, dim3(1), dim3(64), 0, s, stat, op);
  return hipGetLastError();
}

hipError_t launch_stat_check_all(unsigned long long* const* stats, int n, int* bad, hipStream_t s) {
  hipLaunchKernelGGL(stat_check_all_kernel, dim3(1), dim3(64), 0, s, stats, n, bad);
  return hipGetLastError();
}

hipError_t launch_measures(int nbins, const MeasArgs& a, hipStream_t s) {
  if (a.nbins != nbins) return hipErrorInvalidValue;
  hipLaunchKernelGGL((measures_kernel<256>), dim3(meas_grid(nbins)), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace ns2d
