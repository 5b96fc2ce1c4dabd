// Single-context reductions: DeviceReduce-order sums and the disk force
// (the device functions live in fg_reduce.h), and the non-reflecting
// boundary, whose ring means are such sums.
#include <atomic>
#include <mutex>

#include "fg_reduce.h"

template <class Src, int CH>
__global__ __launch_bounds__(RED_TPB) void k_dreduce_partial(Src src, long n, int B, double *partial) {
  dreduce_block<Src, CH>(src, n, B, blockIdx.x, partial);
}

__global__ void k_dreduce_final(const double *partial, int B, double *out, int two, int add_inner) {
  dreduce_final(partial, B, out, two, add_inner);
}

template <class Src>
static fg_status dreduce(fg_ctx *c, Src src, long n, double *out_dev, int two, int add_inner) {
  int B = red_blocks(n);
  // 16 summand rows per round: 8, 24 or 48 measured slower (more rounds, or
  // fewer resident workgroups)
  hipLaunchKernelGGL((k_dreduce_partial<Src, RED_CH>), dim3(B), dim3(RED_TPB), 0, c->stream, src, n, B,
                     c->red_partial);
  FG_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_dreduce_final, dim3(1), dim3(256), 0, c->stream, c->red_partial, B, out_dev, two, add_inner);
  FG_LAUNCH_CHECK();
  return FG_OK;
}

// DeviceReduce of one ring of n <= 8192 values (global memory or LDS) by one
// workgroup: block b of the original takes elements 64 b + t and 64 b + t + 32
// (64 B is at least n, so one round), a half-wave each here, and thread 0 adds
// the blocks that have elements in order.  part: LDS, n / 64 + 1 values.  The
// result is thread 0's.
__device__ __forceinline__ double ring_dreduce(const double *a, int n, double *part) {
  const int t = threadIdx.x & 31, nb = (n + 63) / 64;
  for (int b = threadIdx.x >> 5; b < nb; b += blockDim.x >> 5) {
    const int e = 64 * b + t;
    double acc = 0.0;
    if (e < n) {
      acc += a[e];
      if (e + 32 < n) acc += a[e + 32];
    }
    for (int off = 16; off > 0; off >>= 1) acc += __shfl_down(acc, off, 32);
    if (t == 0) part[b] = acc;
  }
  __syncthreads();
  return threadIdx.x == 0 ? seq_sum_lds(part, nb) : 0.0;
}

__global__ __launch_bounds__(1024) void k_ring_sum(const double *ring, int n, double *out) {
  __shared__ double part[129];
  const double s = ring_dreduce(ring, n, part);
  if (threadIdx.x == 0) *out = s;
}

fg_status fg_ring_sum_async(fg_ctx *c, const double *ring, double *out_dev) {
  hipLaunchKernelGGL(k_ring_sum, dim3(1), dim3(1024), 0, c->stream, ring, c->ns, out_dev);
  FG_LAUNCH_CHECK();
  return FG_OK;
}

double fg_lost_mass_result(const fg_ctx *c) { return c->h_out[2]; }
// of fg_routine_results: the disk force on the star (k < 0) or planet k
void fg_disk_force_result(const fg_ctx *c, int k, double out2[2]) {
  const double *h = c->h_out + (k < 0 ? 0 : FG_OUT_PF + 2 * k);
  out2[0] = h[0];
  out2[1] = h[1];
}

extern "C" fg_status fg_disk_force(fg_ctx *c, double x, double y, double rsmoothing, double *out2) {
  if (!c || !out2) {
    fg_set_error("fg_disk_force: NULL argument");
    return FG_E_INVALID;
  }
  force_src src{c->f[FG_DENS], c->t.Surf, c->t.Rmed, c->t.cos_cell, c->t.sin_cell, x, y, rsmoothing, c->ns};
  if (fg_status s = dreduce(c, src, (long)c->nr * c->ns, c->red_out, 1, 1)) return s;
  FG_HIP(hipStreamSynchronize(c->stream));
  out2[0] = c->h_out[0];
  out2[1] = c->h_out[1];
  return FG_OK;
}

// ---- ComputeForce with the Hill cut (Force.cu:102-135) ---------------
// All dimfxy variants in one launch (blockIdx.y = k), each replaying the
// four DeviceReduce calls of Force.cu:120-123; the final pass adds each of
// the 4 * dimfxy block-sum rows in order into the GlobalForce layout
// [k + o * dimfxy], o = fxi, fxo, fyi, fyo.
__global__ __launch_bounds__(RED_TPB) void k_hill_partial(hill_force_src src, long n, int B, double *partial) {
  const int k = blockIdx.y;
  dreduce_block4(src, k, n, B, blockIdx.x, partial + (long)4 * k * B);
}

__global__ void k_hill_final(const double *partial, int B, int dimfxy, double *out) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;  // row k * 4 + o
  if (r >= 4 * dimfxy) return;
  const double *p = partial + (long)r * B;
  double s = 0.0;
  for (int b = 0; b < B; b++) s += p[b];
  out[(r & 3) * dimfxy + (r >> 2)] = s;
}

extern "C" fg_status fg_disk_force_hill(fg_ctx *c, double x, double y, double rsmoothing, int dimfxy, double a,
                                        double rh, double *globalforce) {
  if (!c || !globalforce) {
    fg_set_error("fg_disk_force_hill: NULL argument");
    return FG_E_INVALID;
  }
  if (dimfxy < 1 || dimfxy > FG_HILL_MAX) {
    fg_set_error("fg_disk_force_hill: dimfxy = %d outside 1..%d", dimfxy, FG_HILL_MAX);
    return FG_E_INVALID;
  }
  const long n = (long)c->nr * c->ns;
  const int B = red_blocks(n);
  if (!c->hill_partial) {
    FG_HIP(hipMalloc((void **)&c->hill_partial, sizeof(double) * 4 * FG_HILL_MAX * FG_RED_BLOCKS));
    FG_HIP(hipMalloc((void **)&c->hill_out, sizeof(double) * 4 * FG_HILL_MAX));
  }
  hill_force_src src{c->f[FG_DENS], c->t.Surf, c->t.Rmed, c->t.cos_cell, c->t.sin_cell, x, y, rsmoothing, a, rh,
                     c->ns, dimfxy};
  hipLaunchKernelGGL(k_hill_partial, dim3(B, dimfxy), dim3(RED_TPB), 0, c->stream, src, n, B, c->hill_partial);
  FG_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_hill_final, dim3((4 * dimfxy + 63) / 64), dim3(64), 0, c->stream, c->hill_partial, B, dimfxy,
                     c->hill_out);
  FG_LAUNCH_CHECK();
  FG_HIP(hipMemcpyAsync(globalforce, c->hill_out, sizeof(double) * 4 * dimfxy, hipMemcpyDeviceToHost, c->stream));
  FG_HIP(hipStreamSynchronize(c->stream));
  return FG_OK;
}

// ---- fg_disk_force_hill without allocation ----------------------------
// The block partials of fg_disk_force_hill_noalloc live in a file-scope
// device array: 4 * FG_HILL_MAX rows of FG_RED_BLOCKS block sums (2 MiB),
// enough for every grid (DeviceReduce never uses more than FG_RED_BLOCKS
// blocks) and every dimfxy <= FG_HILL_MAX.  Each GPU holds its own copy
// until the process ends.  On the host the array's name is not a device
// address: fg_noalloc_setup (called by fg_create with the context's device
// current) asks hipGetSymbolAddress for this device's copy once and keeps
// the pointer; kernels only ever receive that pointer.  Nothing in it needs
// clearing: k_hill_partial writes every row and block k_hill_final reads.
// All calls on one GPU share the array, so calls that overlap on one GPU
// (two streams, two threads) race.
#define FG_NOALLOC_DOUBLES (4 * FG_HILL_MAX * FG_RED_BLOCKS)
#define FG_NOALLOC_DEVICES 64
static __device__ __align__(256) double scratch[FG_NOALLOC_DOUBLES];
static std::atomic<double *> g_scratch_dev[FG_NOALLOC_DEVICES];
static std::mutex g_scratch_mu;

fg_status fg_noalloc_setup(int device) {
  if (device < 0 || device >= FG_NOALLOC_DEVICES) {
    fg_set_error("device %d beyond the %d the allocation-free entry point supports", device, FG_NOALLOC_DEVICES);
    return FG_E_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_dev[device].load()) return FG_OK;
  void *p = nullptr;
  hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    fg_set_error("hipGetSymbolAddress(scratch) on device %d: %s", device, hipGetErrorString(e));
    return FG_E_HIP;
  }
  g_scratch_dev[device].store((double *)p);
  return FG_OK;
}

extern "C" fg_status fg_disk_force_hill_noalloc(fg_ctx *c, double x, double y, double rsmoothing, int dimfxy,
                                                double a, double rh, double *globalforce_dev) {
  if (!c || !globalforce_dev) {
    fg_set_error("fg_disk_force_hill_noalloc: NULL argument");
    return FG_E_INVALID;
  }
  if (dimfxy < 1 || dimfxy > FG_HILL_MAX) {
    fg_set_error("fg_disk_force_hill_noalloc: dimfxy = %d outside 1..%d (the scratch array holds %d variants)",
                 dimfxy, FG_HILL_MAX, FG_HILL_MAX);
    return FG_E_INVALID;
  }
  double *scr = (c->device >= 0 && c->device < FG_NOALLOC_DEVICES) ? g_scratch_dev[c->device].load() : nullptr;
  if (!scr) {
    fg_set_error("fg_disk_force_hill_noalloc: fg_create could not locate the scratch array on device %d",
                 c->device);
    return FG_E_HIP;
  }
  const long n = (long)c->nr * c->ns;
  const int B = red_blocks(n);
  if ((long)4 * dimfxy * B > FG_NOALLOC_DOUBLES) {
    fg_set_error("fg_disk_force_hill_noalloc: %d x %d partial sums exceed the %d-double scratch array", 4 * dimfxy,
                 B, FG_NOALLOC_DOUBLES);
    return FG_E_INVALID;
  }
  hill_force_src src{c->f[FG_DENS], c->t.Surf, c->t.Rmed, c->t.cos_cell, c->t.sin_cell, x, y, rsmoothing, a, rh,
                     c->ns, dimfxy};
  hipLaunchKernelGGL(k_hill_partial, dim3(B, dimfxy), dim3(RED_TPB), 0, c->stream, src, n, B, scr);
  FG_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_hill_final, dim3((4 * dimfxy + 63) / 64), dim3(64), 0, c->stream, scr, B, dimfxy,
                     globalforce_dev);
  FG_LAUNCH_CHECK();
  return FG_OK;
}

// ---- CircumPlanetaryMass (SourceEuler.cu:549-563) --------------------
fg_status fg_circumplanetary_mass_async(fg_ctx *c, double xpl, double ypl, double hill_radius, double *out_dev) {
  cpm_src src{c->f[FG_DENS], c->t.Surf, c->t.Rmed, c->t.cos_cell, c->t.sin_cell, xpl, ypl, hill_radius, c->ns};
  return dreduce(c, src, (long)c->nr * c->ns, out_dev, 0, 0);
}

extern "C" fg_status fg_circumplanetary_mass(fg_ctx *c, double xpl, double ypl, double hill_radius, double *out) {
  if (!c || !out) {
    fg_set_error("fg_circumplanetary_mass: NULL argument");
    return FG_E_INVALID;
  }
  if (fg_status s = fg_circumplanetary_mass_async(c, xpl, ypl, hill_radius, c->red_out + 3)) return s;
  FG_HIP(hipStreamSynchronize(c->stream));
  *out = c->h_out[3];
  return FG_OK;
}

// ---- non-reflecting boundary (SideEuler.cu:45-100) -------------------
// One workgroup per edge does all of it: the ring means of c_s (each
// DeviceReduce(...)/NSEC of SideEuler.cu:84-99 over one ring) and the shift
// they give, the edge ring of Sigma and energy copied shifted from its
// neighbour (Kernels.cu:534-573, wrapped modulo NSEC) and brought to its
// initial mean (Kernels.cu:592-607), and vrad (Kernels.cu:575-589, bounded to
// j < NSEC).  The two edges touch different rings from NRAD = 4 on; a disk of
// three rings runs them one after the other.  Bound: a dozen dependent
// barriers and memory round trips.  As one launch per ring sum and copy, with
// the host computing the shifts, a boundary pass was 22 launches and four
// waits; this is 13 us at NSEC = 1152, and a 384 x 1152 substep with three of
// them takes 166 us with it, fg_transport's sweeps and k_cells, was 880.
struct nr_args {
  double *dens, *energy, *vr, *press, *temp;  // press, temp: NULL or formed anew on the edge rings
  const double *cs, *fpress;
  // inner, outer edge: pow(Rinf, -1.5) - 1 and the ring spacing of the shift's
  // angle, Sigma of vrad's ring, Sigma and energy means of the edge ring
  double num[2], width[2], sigma_v[2], sigma0[2], energy0[2];
  double gamma;
  int nr, ns, adiabatic;
};

// (int)x as the host converts it: out of range and NaN give INT_MIN
__device__ __forceinline__ int nr_to_int(double x) {
  return (x > -2147483649.0 && x < 2147483648.0) ? (int)x : (int)0x80000000;
}

__device__ __forceinline__ void nr_edge(const nr_args &a, int edge, double *ring, double *part) {
  __shared__ double s_sum[2];
  const int nr = a.nr, ns = a.ns, tid = threadIdx.x;
  // rings of the edge, its neighbour, and the one whose vrad is reflected
  const long e = edge ? nr - 1 : 0, n = edge ? nr - 2 : 1;
  for (int q = 0; q < 2; q++) {  // c_s means, in the order of SideEuler.cu
    const double s = ring_dreduce(a.cs + (q ? n : e) * ns, ns, part);
    if (tid == 0) s_sum[q] = s / ns;
    __syncthreads();
  }
  double dangle = a.num[edge] / (.5 * (s_sum[0] + s_sum[1]));
  dangle *= a.width[edge];
  const int shift = nr_to_int(dangle / 2.0 / FG_PI * (double)ns + .5);
  for (int f = 0; f < 2; f++) {
    double *q = f ? a.energy : a.dens;
    __syncthreads();
    for (int j = tid; j < ns; j += blockDim.x) {
      if (edge == 0)
        ring[((j + shift) % ns + ns) % ns] = q[n * ns + j];
      else
        ring[j] = q[n * ns + ((j - shift) % ns + ns) % ns];
    }
    __syncthreads();
    const double s = ring_dreduce(ring, ns, part);
    if (tid == 0) s_sum[0] = s / ns;
    __syncthreads();
    const double add = (f ? a.energy0[edge] : a.sigma0[edge]) - s_sum[0];
    for (int j = tid; j < ns; j += blockDim.x) q[e * ns + j] = ring[j] + add;
  }
  if (a.press || a.temp) {
    for (int j = tid; j < ns; j += blockDim.x) {  // as k_cells, of the cells that this thread wrote
      const long l = e * ns + j;
      if (a.press) a.press[l] = a.adiabatic ? (a.gamma - 1.0) * a.energy[l] : a.dens[l] * a.cs[l] * a.cs[l];
      if (a.temp)
        a.temp[l] = a.adiabatic ? (a.gamma - 1.0) * a.energy[l] / a.dens[l] : a.fpress[l] / a.dens[l];
    }
  }
  const double sm = a.sigma_v[edge];
  for (int j = tid; j < ns; j += blockDim.x) {
    if (edge == 0) {
      const double Vrad_med = -a.cs[ns + j] * (a.dens[ns + j] - sm) / sm;
      a.vr[ns + j] = 2.0 * Vrad_med - a.vr[2L * ns + j];
    } else {
      const long i = nr - 1;
      const double Vrad_med = a.cs[i * ns + j] * (a.dens[(i - 1) * ns + j] - sm) / sm;
      a.vr[i * ns + j] = 2. * Vrad_med - a.vr[(i - 1) * ns + j];
    }
  }
}

__global__ __launch_bounds__(1024) void k_nr_edges(nr_args a) {
  extern __shared__ double ring[];
  __shared__ double part[129];
  if (gridDim.x == 2) {
    nr_edge(a, blockIdx.x, ring, part);
  } else {
    nr_edge(a, 0, ring, part);
    __syncthreads();
    nr_edge(a, 1, ring, part);
  }
}

void fg_ask_edge_lds() {
  (void)hipFuncSetAttribute((const void *)k_nr_edges, hipFuncAttributeMaxDynamicSharedMemorySize, FG_RING_LDS);
}

fg_status fg_nonreflecting_internal(fg_ctx *c, double *press, double *temp) {
  const int nr = c->nr, ns = c->ns;
  const std::vector<double> &Rinf = c->h_Rinf, &Rmed = c->h_Rmed;
  nr_args a;
  a.dens = c->f[FG_DENS];
  a.energy = c->f[FG_ENERGY];
  a.vr = c->f[FG_VRAD];
  a.cs = c->f[FG_SOUNDSPEED];
  a.press = press;
  a.temp = temp;
  a.fpress = c->f[FG_PRESSURE];
  a.gamma = c->p.adiabatic_index;
  a.adiabatic = c->p.adiabatic;
  a.num[0] = pow(Rinf[1], -1.5) - 1.0;
  a.width[0] = Rmed[1] - Rmed[0];
  a.num[1] = pow(Rinf[nr - 2], -1.5) - 1.0;
  a.width[1] = Rmed[nr - 1] - Rmed[nr - 2];
  a.sigma_v[0] = c->h_SigmaMed[1];
  a.sigma_v[1] = c->h_SigmaMed[nr - 2];
  a.sigma0[0] = c->h_SigmaMed[0];
  a.sigma0[1] = c->h_SigmaMed[nr - 1];
  a.energy0[0] = c->h_EnergyMed[0];
  a.energy0[1] = c->h_EnergyMed[nr - 1];
  a.nr = nr;
  a.ns = ns;
  hipLaunchKernelGGL(k_nr_edges, dim3(nr > 3 ? 2 : 1), dim3(1024), (size_t)ns * sizeof(double), c->stream, a);
  FG_LAUNCH_CHECK();
  return FG_OK;
}
