// Batched (segmented) Jacobi-preconditioned CG for many independent
// systems of uneven size: one launch per CG phase serves every system in
// the batch, and a fixed number of iterations is captured once into a
// hipGraph that is replayed while systems join and leave (the graph's
// kernels read the current systems from device tables, so membership
// changes need no re-capture).
//
// Each system's rows are cut into chunks of a fixed number of rows that
// depends only on the system, reductions are summed per system in chunk
// order, and nothing is shared between systems: a system's iterates are
// bitwise the same alone and in any mix. gfx950 (MI355X) only.
#include "device.hpp"

#include <algorithm>
#include <cstring>
#include <vector>

namespace dfx
{
namespace
{

constexpr int kBlock = 256;
constexpr int kLanes = 4;                // lanes per row (P1 rows ~15)
constexpr int kSteps = 4;                // entries per lane loaded together
constexpr int kRowsPerPass = kBlock / kLanes;
// Rows per chunk. A chunk is the unit of the reductions (one partial per
// chunk), so its size fixes how many partials every workgroup re-sums: with
// 64 rows the 117,649 rows of a 48^3 mesh had 1,839 partials re-summed for
// every chunk, and 64 of the 256 threads had a row in the vector phases
// (update 33 us, direction 31 us for sixteen systems of 8^3 to 48^3); with
// 256 rows every thread has one and a workgroup sums 460 partials once.
constexpr int kRowsPerChunk = 256;

/// Device view of one system (FP64).
struct SysDesc
{
  const std::int32_t* rp;
  const std::int32_t* ci;
  const double* v;
  const double* b;
  double* x;
  double* r;
  double* p;
  double* q;
  double* dinv;
  double2* zp; // per row (z, previous p): what the next SpMV gathers
  const std::int32_t* diag; // CSR position of each row's diagonal (-1: none)
  std::int32_t nrows;
  std::int32_t chunk0; // first chunk of the system
  std::int32_t nchunks;
  std::int32_t pad;
};

/// Per-system CG scalars. The SpMV phase of iteration k reads k from
/// iter_next and writes iter, the update phase reads iter and writes
/// iter_next, so no kernel writes what another of its workgroups reads
/// (done excepted: it is only ever set by the workgroup whose decision the
/// others reach from the same sums).
struct SysState
{
  double rz[2];
  double rr0, rr, tol2;
  std::int32_t iter, iter_next, done, max_it;
  std::int32_t active, converged;
  // iteration whose stop test and rz are in the state already (set at the
  // start and after the last iteration of a step: the partials move when
  // systems join or leave between steps)
  std::int32_t tested, pad;
};

struct ChunkDesc
{
  std::int32_t sys, row0, row1, first; // first: chunk is the system's first
};

/// Chunks of one workgroup: a contiguous range, and contiguous over the
/// workgroups of an XCD, so that a system's partials are summed once per
/// workgroup (not once per chunk) and both phases find their rows in the
/// same L2.
__device__ inline int2 chunk_range(int nch)
{
  const int nb = gridDim.x;
  const int l = xcd_contiguous(blockIdx.x, nb);
  return {static_cast<int>(static_cast<long long>(nch) * l / nb),
          static_cast<int>(static_cast<long long>(nch) * (l + 1) / nb)};
}

/// Whether a system takes no part in this phase, read once per block so that
/// every wavefront of the block takes the same branch.
__device__ inline bool block_skip(const SysState& S)
{
  __shared__ int skip;
  if (threadIdx.x == 0)
    skip = (__hip_atomic_load(&S.active, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0
            || __hip_atomic_load(&S.done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
               ? 1
               : 0;
  __syncthreads();
  const bool r = skip != 0;
  __syncthreads();
  return r;
}

/// Stop test of a system before iteration k (k >= 1) from the reductions of
/// the iterations so far.
__device__ inline bool stop_test(const SysState& S, int k, double rr, bool& conv)
{
  conv = rr / S.rr0 < S.tol2;
  return conv || k >= S.max_it;
}

/// First phase of iteration k: stop test and beta from the last update's
/// sums, p = z + beta p formed where it is gathered (each row's z and
/// previous p are one 16-byte load), q = A p and the partial sums of p . q.
/// Two kernels per iteration instead of three (SpMV, update, direction): the
/// bytes are the same (the direction kernel's reads of r, dinv and p became
/// the pair), a launch and a pass of latency are gone. Four lanes per row,
/// the first 4 x kSteps entries of two rows per thread loaded before their
/// gathers. Sixteen systems of 8^3 to 48^3 (618,000 rows, 8.8 M entries,
/// 106 MB of matrix: it stays in the on-package cache): 41 us per iteration
/// (31 here, 10 in the update) against 99.5 us of the three kernels; the
/// whole wave of requests 14.8 ms against 27.0 ms.
__global__ void __launch_bounds__(kBlock)
    bcg_spmv_k(const int* nchunk, const ChunkDesc* chunks, const SysDesc* sys, SysState* st,
               double* p_pq, const double* p_rz, const double* p_rr)
{
  const int2 range = chunk_range(*nchunk);
  int cur = -1;
  bool skip = false;
  double beta = 0;
  for (int t = range.x; t < range.y; ++t)
  {
    const ChunkDesc ch = chunks[t];
    const SysDesc& D = sys[ch.sys];
    if (ch.sys != cur)
    {
      cur = ch.sys;
      SysState& S = st[cur];
      skip = block_skip(S);
      if (!skip)
      {
        const int k = S.iter_next;
        if (S.tested == k)
          beta = k > 0 ? S.rz[k & 1] / S.rz[(k - 1) & 1] : 0.0;
        else
        {
          double sums[2];
          sum_ranges<2>({p_rz, p_rr}, D.chunk0, D.nchunks, sums);
          bool conv;
          skip = stop_test(S, k, sums[1], conv);
          beta = sums[0] / S.rz[(k - 1) & 1];
          if (ch.first && threadIdx.x == 0)
          {
            S.rz[k & 1] = sums[0];
            S.rr = sums[1];
            if (skip)
            {
              S.converged = conv ? 1 : 0;
              __hip_atomic_store(&S.done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
          }
        }
        if (ch.first && threadIdx.x == 0)
          S.iter = k;
      }
    }
    if (skip)
      continue;
    const int lane = threadIdx.x % kLanes;
    const std::int32_t* __restrict__ ci = D.ci;
    const double* __restrict__ v = D.v;
    const double2* __restrict__ zp = D.zp;
    double d = 0;
#pragma unroll
    for (int half = 0; half < kRowsPerChunk / kRowsPerPass; half += 2)
    {
      std::int32_t row[2], e[2], c[2][kSteps];
      std::int32_t j[2];
      double a[2][kSteps];
      double2 own[2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
      {
        row[h] = ch.row0 + (half + h) * kRowsPerPass + threadIdx.x / kLanes;
        const std::int32_t rr = min(row[h], ch.row1 - 1);
        j[h] = D.rp[rr] + lane;
        e[h] = D.rp[rr + 1];
        own[h] = zp[rr];
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < kSteps; ++i)
        {
          // past the row's end: its last entry again, added as zero
          const std::int32_t jj = max(min(j[h] + i * kLanes, e[h] - 1), 0);
          c[h][i] = ci[jj];
          a[h][i] = v[jj];
        }
      double s[2] = {0, 0};
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < kSteps; ++i)
        {
          const double2 g = zp[c[h][i]];
          if (j[h] + i * kLanes < e[h])
            s[h] += a[h][i] * __builtin_fma(beta, g.y, g.x);
        }
#pragma unroll
      for (int h = 0; h < 2; ++h)
      {
        for (std::int32_t q = j[h] + kSteps * kLanes; q < e[h]; q += kLanes)
        {
          const double2 g = zp[ci[q]];
          s[h] += v[q] * __builtin_fma(beta, g.y, g.x);
        }
#pragma unroll
        for (int off = kLanes / 2; off > 0; off >>= 1)
          s[h] += __shfl_down(s[h], off, kLanes);
        if (lane == 0 && row[h] < ch.row1)
        {
          const double p = __builtin_fma(beta, own[h].y, own[h].x);
          D.p[row[h]] = p;
          D.q[row[h]] = s[h];
          d += s[h] * p;
        }
      }
    }
    store_block_sums<1>({d}, {p_pq}, t);
  }
}

/// Second phase: x += alpha p, r -= alpha q, the pairs (dinv r, p) that the
/// next SpMV gathers, and the partial sums of r . z and r . r.
__global__ void __launch_bounds__(kBlock)
    bcg_update_k(const int* nchunk, const ChunkDesc* chunks, const SysDesc* sys, SysState* st,
                 const double* p_pq, double* p_rz, double* p_rr)
{
  const int2 range = chunk_range(*nchunk);
  int cur = -1;
  bool skip = false;
  double alpha = 0;
  for (int t = range.x; t < range.y; ++t)
  {
    const ChunkDesc ch = chunks[t];
    const SysDesc& D = sys[ch.sys];
    if (ch.sys != cur)
    {
      cur = ch.sys;
      SysState& S = st[cur];
      skip = block_skip(S);
      if (!skip)
      {
        double pq[1];
        sum_ranges<1>({p_pq}, D.chunk0, D.nchunks, pq);
        const int k = S.iter;
        alpha = S.rz[k & 1] / pq[0];
        if (ch.first && threadIdx.x == 0)
          S.iter_next = k + 1;
      }
    }
    if (skip)
      continue;
    double sums[2] = {0, 0};
    const std::int32_t i = ch.row0 + threadIdx.x;
    if (i < ch.row1)
    {
      const double p = D.p[i], di = D.dinv[i];
      D.x[i] += alpha * p;
      const double ri = D.r[i] - alpha * D.q[i];
      D.r[i] = ri;
      const double z = di * ri;
      D.zp[i] = make_double2(z, p);
      sums[0] = z * ri;
      sums[1] = ri * ri;
    }
    store_block_sums<2>(sums, {p_rz, p_rr}, t);
  }
}

/// After the last iteration of a step: the stop test and r . z that the next
/// SpMV would take from the partials, so that the status read then is that of
/// every iteration done and the partials are free to move.
__global__ void __launch_bounds__(kBlock)
    bcg_finish_k(int nsys, const SysDesc* sys, SysState* st, const double* p_rz,
                 const double* p_rr)
{
  for (int s = blockIdx.x; s < nsys; s += gridDim.x)
  {
    SysState& S = st[s];
    if (block_skip(S) || S.tested == S.iter_next)
      continue;
    const SysDesc& D = sys[s];
    double sums[2];
    sum_ranges<2>({p_rz, p_rr}, D.chunk0, D.nchunks, sums); // ends with a barrier
    if (threadIdx.x == 0)
    {
      bool conv;
      const int k = S.iter_next;
      S.rz[k & 1] = sums[0];
      S.rr = sums[1];
      S.tested = k;
      if (stop_test(S, k, sums[1], conv))
      {
        S.converged = conv ? 1 : 0;
        S.done = 1;
      }
    }
    __syncthreads();
  }
}

/// First residual of one row: r = b, z = dinv b, x = 0 (dinv from the CSR
/// diagonal); adds its r . z and r . r to sums.
__device__ inline void start_row(const SysDesc& D, const std::int32_t* diag, std::int32_t i,
                                 double (&sums)[2])
{
  const std::int32_t pd = diag[i];
  const double a = pd >= 0 ? D.v[pd] : 0.0;
  const double di = a != 0.0 ? 1.0 / a : 1.0;
  const double bi = D.b[i];
  D.dinv[i] = di;
  D.x[i] = 0.0;
  D.r[i] = bi;
  const double z = di * bi;
  D.zp[i] = make_double2(z, 0.0);
  sums[0] += z * bi;
  sums[1] += bi * bi;
}

/// Start of a system's solve from x = 0: start_row and the partial sums.
__global__ void __launch_bounds__(kBlock)
    bcg_start_k(SysDesc D, const std::int32_t* diag, int c0, double* p_rz, double* p_rr)
{
  const std::int32_t i = blockIdx.x * kRowsPerChunk + threadIdx.x;
  double sums[2] = {0, 0};
  if (i < D.nrows)
    start_row(D, diag, i, sums);
  store_block_sums<2>(sums, {p_rz, p_rr}, c0 + blockIdx.x);
}

__device__ inline void start_state(SysState& S, const double (&sums)[2])
{
  S.rz[0] = sums[0];
  S.rz[1] = 0;
  S.rr0 = sums[1];
  S.rr = sums[1];
  S.iter = 0;
  S.iter_next = 0;
  S.tested = 0;
  S.converged = sums[1] == 0.0 ? 1 : 0;
  S.done = (sums[1] == 0.0 || S.max_it <= 0) ? 1 : 0;
}

__global__ void __launch_bounds__(kBlock)
    bcg_start_finish_k(const double* p_rz, const double* p_rr, int c0, int n, SysState* S,
                       double tol2, int max_it)
{
  double sums[2];
  sum_ranges<2>({p_rz, p_rr}, c0, n, sums);
  if (threadIdx.x == 0)
  {
    S->tol2 = tol2;
    S->max_it = max_it;
    S->active = 1;
    start_state(*S, sums);
  }
}

/// Restart of every active system from x = 0, chunk by chunk over the
/// batch's tables (the values of bcg_start_k for each chunk).
__global__ void __launch_bounds__(kBlock)
    bcg_restart_k(const int* nchunk, const ChunkDesc* chunks, const SysDesc* sys,
                  const SysState* st, double* p_rz, double* p_rr)
{
  const int2 range = chunk_range(*nchunk);
  for (int t = range.x; t < range.y; ++t)
  {
    const ChunkDesc ch = chunks[t];
    if (st[ch.sys].active == 0)
      continue;
    const SysDesc& D = sys[ch.sys];
    double sums[2] = {0, 0};
    const std::int32_t i = ch.row0 + threadIdx.x;
    if (i < ch.row1)
      start_row(D, D.diag, i, sums);
    store_block_sums<2>(sums, {p_rz, p_rr}, t);
  }
}

/// Per system (one workgroup per slot): the restart's reductions and
/// counters, as bcg_start_finish_k with the system's rtol and max_it kept.
__global__ void __launch_bounds__(kBlock)
    bcg_restart_finish_k(int nsys, const SysDesc* sys, SysState* st, const double* p_rz,
                         const double* p_rr)
{
  for (int s = blockIdx.x; s < nsys; s += gridDim.x)
  {
    SysState& S = st[s];
    if (S.active == 0)
      continue;
    const SysDesc& D = sys[s];
    double sums[2];
    sum_ranges<2>({p_rz, p_rr}, D.chunk0, D.nchunks, sums);
    if (threadIdx.x == 0)
      start_state(S, sums);
    __syncthreads();
  }
}

} // namespace
} // namespace dfx

using namespace dfx;

/// A batch of independent FP64 CG solves.
struct dfx_batch
{
  std::int32_t max_sys = 0, max_chunks = 0;
  std::vector<SysDesc> hsys;
  std::vector<int> slot_used;
  std::vector<std::int32_t> chunks_of; // per slot
  SysDesc* sys = nullptr;
  SysState* st = nullptr;
  ChunkDesc* chunks = nullptr;
  int* nchunk = nullptr;
  double* p_pq = nullptr;
  double* p_rz = nullptr;
  double* p_rr = nullptr;
  // graph of `graph_iters` iterations
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int graph_iters = 0;
  // work vectors (r, p, q, diag^-1, (z, p) pairs) of systems that left, kept by row count
  // for the next system of that size (no device allocation or free, and so
  // no device-wide synchronisation, while serving)
  struct Work
  {
    std::int64_t n;
    double* v[5];
  };
  std::vector<Work> pool;
};

namespace
{

void batch_rebuild_chunks(dfx_batch& B)
{
  no_capture("a change of batch membership");
  std::vector<ChunkDesc> ch;
  for (int s = 0; s < B.max_sys; ++s)
  {
    if (!B.slot_used[s])
      continue;
    SysDesc& d = B.hsys[s];
    d.chunk0 = static_cast<std::int32_t>(ch.size());
    d.nchunks = (d.nrows + kRowsPerChunk - 1) / kRowsPerChunk;
    for (int c = 0; c < d.nchunks; ++c)
      ch.push_back({s, c * kRowsPerChunk, std::min((c + 1) * kRowsPerChunk, d.nrows), c == 0});
  }
  require(static_cast<int>(ch.size()) <= B.max_chunks, "batch is full (rows)");
  const int n = static_cast<int>(ch.size());
  if (n)
    DFX_HIP(hipMemcpyAsync(B.chunks, ch.data(), sizeof(ChunkDesc) * n, hipMemcpyHostToDevice, stream()));
  DFX_HIP(hipMemcpyAsync(B.nchunk, &n, sizeof(int), hipMemcpyHostToDevice, stream()));
  DFX_HIP(hipMemcpyAsync(B.sys, B.hsys.data(), sizeof(SysDesc) * B.max_sys, hipMemcpyHostToDevice,
                         stream()));
  DFX_HIP(hipStreamSynchronize(stream()));
}

/// Workgroups of the phase kernels: a fixed grid (so that a captured graph
/// stays valid) striding over the live chunks.
int phase_grid(const dfx_batch& B)
{
  return std::max(1, std::min(B.max_chunks, ctx().num_cu * 8));
}

void launch_iterations(dfx_batch& B, int iters)
{
  hipStream_t s = stream();
  const int g = phase_grid(B);
  for (int i = 0; i < iters; ++i)
  {
    bcg_spmv_k<<<g, kBlock, 0, s>>>(B.nchunk, B.chunks, B.sys, B.st, B.p_pq, B.p_rz, B.p_rr);
    bcg_update_k<<<g, kBlock, 0, s>>>(B.nchunk, B.chunks, B.sys, B.st, B.p_pq, B.p_rz, B.p_rr);
  }
  bcg_finish_k<<<std::min(B.max_sys, 1024), kBlock, 0, s>>>(B.max_sys, B.sys, B.st, B.p_rz,
                                                           B.p_rr);
}

} // namespace

extern "C" {

dfx_status dfx_batch_create(int32_t max_systems, int64_t max_rows, dfx_batch** out)
{
  return guard(
      [&]
      {
        require(out && max_systems > 0 && max_rows > 0, "bad argument");
        auto B = std::make_unique<dfx_batch>();
        B->max_sys = max_systems;
        B->max_chunks = static_cast<std::int32_t>((max_rows + kRowsPerChunk - 1) / kRowsPerChunk
                                                  + max_systems);
        B->hsys.assign(max_systems, SysDesc{});
        B->slot_used.assign(max_systems, 0);
        B->sys = static_cast<SysDesc*>(dmalloc(sizeof(SysDesc) * max_systems));
        B->st = static_cast<SysState*>(dmalloc(sizeof(SysState) * max_systems));
        B->chunks = static_cast<ChunkDesc*>(dmalloc(sizeof(ChunkDesc) * B->max_chunks));
        B->nchunk = static_cast<int*>(dmalloc(sizeof(int)));
        B->p_pq = static_cast<double*>(dmalloc(sizeof(double) * B->max_chunks));
        B->p_rz = static_cast<double*>(dmalloc(sizeof(double) * B->max_chunks));
        B->p_rr = static_cast<double*>(dmalloc(sizeof(double) * B->max_chunks));
        DFX_HIP(hipMemsetAsync(B->st, 0, sizeof(SysState) * max_systems, stream()));
        batch_rebuild_chunks(*B);
        *out = B.release();
      });
}

dfx_status dfx_batch_destroy(dfx_batch* B)
{
  if (B)
  {
    if (B->exec)
      (void)hipGraphExecDestroy(B->exec);
    if (B->graph)
      (void)hipGraphDestroy(B->graph);
    for (int s = 0; s < B->max_sys; ++s)
      if (B->slot_used[s])
      {
        dfree(B->hsys[s].r);
        dfree(B->hsys[s].p);
        dfree(B->hsys[s].q);
        dfree(B->hsys[s].dinv);
        dfree(B->hsys[s].zp);
      }
    for (auto& w : B->pool)
      for (double* v : w.v)
        dfree(v);
    dfree(B->sys);
    dfree(B->st);
    dfree(B->chunks);
    dfree(B->nchunk);
    dfree(B->p_pq);
    dfree(B->p_rz);
    dfree(B->p_rr);
    delete B;
  }
  return DFX_OK;
}

dfx_status dfx_batch_add(dfx_batch* B, const dfx_csr* A, const dfx_vec* b, dfx_vec* x,
                         double rtol, int32_t max_it, int32_t* slot)
{
  return guard(
      [&]
      {
        require(B && A && b && x && slot, "null argument");
        require(A->dtype == DFX_F64 && b->dtype == DFX_F64 && x->dtype == DFX_F64,
                "batched CG runs in FP64");
        require(A->bs == 1 && A->nrows == A->ncols, "scalar square matrix required");
        require(b->n == A->nrows && x->n == A->nrows, "size mismatch");
        int s = -1;
        for (int i = 0; i < B->max_sys; ++i)
          if (!B->slot_used[i])
          {
            s = i;
            break;
          }
        require(s >= 0, "batch is full (systems)");
        materialize_zero(*A);
        SysDesc d{};
        d.rp = A->row_ptr;
        d.ci = A->cols;
        d.v = static_cast<const double*>(A->values);
        d.b = static_cast<const double*>(b->data);
        d.x = static_cast<double*>(x->data);
        d.diag = A->diag;
        d.nrows = A->nrows;
        const std::int64_t n = std::max(A->nrows, 1);
        auto it = std::find_if(B->pool.begin(), B->pool.end(),
                               [&](const dfx_batch::Work& w) { return w.n == n; });
        if (it != B->pool.end())
        {
          d.r = it->v[0];
          d.p = it->v[1];
          d.q = it->v[2];
          d.dinv = it->v[3];
          d.zp = reinterpret_cast<double2*>(it->v[4]);
          B->pool.erase(it);
        }
        else
        {
          d.r = static_cast<double*>(dmalloc(sizeof(double) * n));
          d.p = static_cast<double*>(dmalloc(sizeof(double) * n));
          d.q = static_cast<double*>(dmalloc(sizeof(double) * n));
          d.dinv = static_cast<double*>(dmalloc(sizeof(double) * n));
          d.zp = static_cast<double2*>(dmalloc(sizeof(double2) * n));
        }
        if (A->nnz == 0)
        {
          // the SpMV loads (and drops) entry 0 for an empty row: give it one
          d.ci = A->row_ptr;
          d.v = d.dinv;
        }
        B->hsys[s] = d;
        B->slot_used[s] = 1;
        try
        {
          batch_rebuild_chunks(*B);
        }
        catch (...)
        {
          B->slot_used[s] = 0;
          dfree(d.r);
          dfree(d.p);
          dfree(d.q);
          dfree(d.dinv);
          dfree(d.zp);
          throw;
        }
        const SysDesc& dd = B->hsys[s];
        if (dd.nrows > 0)
          bcg_start_k<<<dd.nchunks, kBlock, 0, stream()>>>(dd, A->diag, dd.chunk0, B->p_rz,
                                                          B->p_rr);
        bcg_start_finish_k<<<1, kBlock, 0, stream()>>>(B->p_rz, B->p_rr, dd.chunk0, dd.nchunks,
                                                       B->st + s, rtol * rtol, max_it);
        check_launch("batch_add");
        *slot = s;
      });
}

dfx_status dfx_batch_remove(dfx_batch* B, int32_t slot)
{
  return guard(
      [&]
      {
        require(B && slot >= 0 && slot < B->max_sys && B->slot_used[slot], "bad slot");
        SysDesc& d = B->hsys[slot];
        // queued work of this system precedes any later use of its vectors
        // in stream order, so they go back to the pool at once
        B->pool.push_back({std::max<std::int64_t>(d.nrows, 1), {d.r, d.p, d.q, d.dinv, reinterpret_cast<double*>(d.zp)}});
        d = SysDesc{};
        B->slot_used[slot] = 0;
        SysState zero{};
        DFX_HIP(hipMemcpyAsync(B->st + slot, &zero, sizeof(SysState), hipMemcpyHostToDevice, stream()));
        batch_rebuild_chunks(*B);
      });
}

dfx_status dfx_batch_step(dfx_batch* B, int32_t iterations, int32_t use_graph)
{
  return guard(
      [&]
      {
        require(B && iterations > 0, "bad argument");
        // inside an open capture the iterations are recorded into it
        if (!use_graph || capturing())
        {
          launch_iterations(*B, iterations);
          check_launch("batch_step");
          return;
        }
        if (!B->exec || B->graph_iters != iterations)
        {
          if (B->exec)
            (void)hipGraphExecDestroy(B->exec);
          if (B->graph)
            (void)hipGraphDestroy(B->graph);
          B->exec = nullptr;
          B->graph = nullptr;
          DFX_HIP(hipStreamBeginCapture(stream(), hipStreamCaptureModeThreadLocal));
          launch_iterations(*B, iterations);
          DFX_HIP(hipStreamEndCapture(stream(), &B->graph));
          DFX_HIP(hipGraphInstantiate(&B->exec, B->graph, nullptr, nullptr, 0));
          B->graph_iters = iterations;
        }
        DFX_HIP(hipGraphLaunch(B->exec, stream()));
      });
}

dfx_status dfx_batch_restart(dfx_batch* B)
{
  return guard(
      [&]
      {
        require(B, "null batch");
        hipStream_t s = stream();
        bcg_restart_k<<<phase_grid(*B), kBlock, 0, s>>>(B->nchunk, B->chunks, B->sys, B->st,
                                                        B->p_rz, B->p_rr);
        bcg_restart_finish_k<<<std::min(B->max_sys, 1024), kBlock, 0, s>>>(
            B->max_sys, B->sys, B->st, B->p_rz, B->p_rr);
        check_launch("batch_restart");
      });
}

dfx_status dfx_batch_status(dfx_batch* B, int32_t n, const int32_t* slots, int32_t* done,
                            int32_t* converged, int32_t* iterations, double* rel_residual)
{
  return guard(
      [&]
      {
        require(B && (n == 0 || slots), "bad argument");
        std::vector<SysState> h(B->max_sys);
        d2h(h.data(), B->st, sizeof(SysState) * B->max_sys);
        for (int i = 0; i < n; ++i)
        {
          require(slots[i] >= 0 && slots[i] < B->max_sys, "bad slot");
          const SysState& S = h[slots[i]];
          if (done)
            done[i] = S.done;
          if (converged)
            converged[i] = S.converged;
          if (iterations)
            iterations[i] = S.iter_next;
          if (rel_residual)
            rel_residual[i] = S.rr0 > 0 ? std::sqrt(S.rr / S.rr0) : 0.0;
        }
      });
}

} // extern "C"
