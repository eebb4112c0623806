// Ragged batch of BP5 problems solved by one device-resident CG per
// problem, replayed from a captured hipGraph. No reference counterpart;
// each problem is set up exactly as bp5_t (BP/BP5/src/bp5Setup.cpp:29-95:
// box mesh, masked ogs, GlobalToLocal) and iterates cg::Solve
// (libs/core/linearSolverCG.cpp:62-129).
//
// Layout (see batch.hip): global vectors concatenated by problem; local
// vectors concatenated by degree group (problems of one degree share one Ax
// launch, their elements back to back); the gather maps of all problems
// concatenated with offsets, so one gather launch serves the batch and each
// row still sums its entries in the reference's ascending order.
#include <algorithm>
#include <cmath>
#include <map>

#include "bpx.hpp"

namespace bpx {

namespace {
constexpr int kChunk = 4096;        // vector entries per streaming workgroup
constexpr int kSuperBlocks = 8;     // row blocks per gather super-block
constexpr int kGraphIters = 8;      // CG iterations per captured graph
}  // namespace

bp_batch_t::~bp_batch_t() {
  // (a call that failed half way may have left work queued)
  if (stream) (void)hipStreamSynchronize(stream);
  if (graphExec) (void)hipGraphExecDestroy(graphExec);
  if (graphMixed) (void)hipGraphExecDestroy(graphMixed);
  if (h_count) (void)hipHostFree(h_count);
  for (auto& e : evCount)
    if (e) (void)hipEventDestroy(e);
  if (ev0) (void)hipEventDestroy(ev0);
  if (ev1) (void)hipEventDestroy(ev1);
  if (stream) (void)hipStreamDestroy(stream);
}

int bp_batch_t::Setup(platform_t& p, const std::vector<MeshOpts>& opts, dfloat lambda_) {
  platform = &p;
  lambda = lambda_;
  nprob = (int)opts.size();
  if (nprob < 1) return set_error(BPX_ERR_INVALID_ARGUMENT, "batch: no problems");
  BPX_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
  BPX_HIP(hipEventCreateWithFlags(&ev0, hipEventDisableTiming));
  BPX_HIP(hipEventCreateWithFlags(&ev1, hipEventDisableTiming));
  for (auto& e : evCount) BPX_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  BPX_HIP(hipHostMalloc((void**)&h_count, 2 * sizeof(int), hipHostMallocDefault));
  if (int st = prepare_box_batch()) return st;

  // ---- per-problem host setup (bp5_t: mesh, masked ogs, GlobalToLocal)
  std::vector<mesh_t> meshes(nprob);
  std::vector<ogs::ogs_t> ogss(nprob);
  std::vector<std::vector<dlong>> g2l(nprob);
  for (int i = 0; i < nprob; ++i) {
    if (opts[i].affine) return set_error(BPX_ERR_UNSUPPORTED, "batch: non-affine (perturbed) meshes only");
    MeshOpts o = opts[i];
    o.cubature = 0;
    if (int st = meshes[i].Setup(o)) return st;
    std::vector<hlong> ids;
    meshes[i].MaskedGlobalIds(1, ids);
    const dlong NL = (dlong)ids.size();
    if (int st = ogss[i].Setup(NL, ids.data())) return st;
    g2l[i].resize(NL);
    ogss[i].SetupGlobalToLocalMapping(g2l[i].data());
  }

  // ---- global offsets (problem order)
  off.assign(nprob + 1, 0);
  for (int i = 0; i < nprob; ++i) {
    const long long next = (long long)off[i] + ogss[i].Ngather;
    if (next >= (1LL << 31)) return set_error(BPX_ERR_UNSUPPORTED, "batch: more than 2^31 unknowns");
    off[i + 1] = (dlong)next;
  }
  Ntot = off[nprob];

  // ---- degree groups; local layout group by group, problems in order
  std::map<int, int> groupOf;
  for (int i = 0; i < nprob; ++i)
    if (!groupOf.count(meshes[i].N)) {
      const int g = (int)groups.size();
      groupOf[meshes[i].N] = g;
      groups.emplace_back();
      groups[g].N = meshes[i].N;
      groups[g].Nq = meshes[i].Nq;
    }
  std::vector<long long> localOff(nprob);  // start of problem i in the local vector
  long long loff = 0;
  for (auto& G : groups) {
    G.loff = loff;
    G.Nel = 0;
    for (int i = 0; i < nprob; ++i)
      if (meshes[i].N == G.N) {
        localOff[i] = loff + (long long)G.Nel * meshes[i].Np;
        G.Nel += meshes[i].Nelements;
      }
    loff += (long long)G.Nel * G.Nq * G.Nq * G.Nq;
  }
  if (loff >= (1LL << 31)) return set_error(BPX_ERR_UNSUPPORTED, "batch: more than 2^31 local nodes");
  NLocalTot = (dlong)loff;

  hipStream_t s = stream;
  for (auto& G : groups) {
    const int Np = G.Nq * G.Nq * G.Nq;
    std::vector<double> ggeo, wJ;
    std::vector<dlong> G2L, pid, list(G.Nel);
    ggeo.reserve((size_t)G.Nel * Np * 6);
    wJ.reserve((size_t)G.Nel * Np);
    G2L.reserve((size_t)G.Nel * Np);
    pid.reserve(G.Nel);
    const std::vector<double>* D = nullptr;
    for (int i = 0; i < nprob; ++i) {
      if (meshes[i].N != G.N) continue;
      const mesh_t& m = meshes[i];
      D = &m.D;
      ggeo.insert(ggeo.end(), m.ggeo.begin(), m.ggeo.end());
      wJ.insert(wJ.end(), m.wJ.begin(), m.wJ.end());
      for (dlong l = 0; l < (dlong)g2l[i].size(); ++l) G2L.push_back(g2l[i][l] >= 0 ? g2l[i][l] + off[i] : -1);
      for (dlong e = 0; e < m.Nelements; ++e) pid.push_back(i);
    }
    for (dlong e = 0; e < G.Nel; ++e) list[e] = e;
    if (int st = G.ggeo.upload(ggeo, s)) return st;
    if (int st = G.wJ.upload(wJ, s)) return st;
    if (int st = G.G2L.upload(G2L, s)) return st;
    if (int st = G.elemPid.upload(pid, s)) return st;
    if (int st = G.elementList.upload(list, s)) return st;
    if (int st = G.D.upload(*D, s)) return st;
  }

  // ---- the box kernels' tables: the elements' map coefficients and the
  // degrees' 1D data, per problem its grid and offsets, per class of degrees
  // the workgroups (high degrees first: theirs run longest)
  std::vector<BoxBatchProb> probs(nprob);
  std::vector<double> geo, tab;
  std::vector<BoxBatchItem> items[2], gitems[2];
  std::vector<Group*> byDegree;
  for (auto& G : groups) byDegree.push_back(&G);
  std::sort(byDegree.begin(), byDegree.end(), [](const Group* a, const Group* b) { return a->N > b->N; });
  int npAp = 0;
  for (Group* G : byDegree) {
    const int epb = box_ax_elements(G->Nq), gepb = box_gather_elements(G->Nq), cls = box_batch_class(G->N);
    const int tab0 = (int)tab.size();
    const mesh_t* any = nullptr;
    G->item0 = (int)items[cls].size();
    for (int i = 0; i < nprob; ++i) {
      const mesh_t& m = meshes[i];
      if (m.N != G->N) continue;
      any = &m;
      BoxBatchProb& pr = probs[i];
      pr.g.set(m.opts.nx, m.opts.ny, m.opts.nz, m.N);
      pr.off = off[i];
      pr.loc = localOff[i];
      pr.el0 = (long long)geo.size() / 24;
      pr.tab = tab0;
      pr.pAp0 = npAp;
      pr.npAp = (m.Nelements + epb - 1) / epb;
      npAp += pr.npAp;
      std::vector<double> c;
      m.TrilinearCoefficients(c);
      geo.insert(geo.end(), c.begin(), c.end());
      for (dlong e = 0; e < m.Nelements; e += epb) items[cls].push_back({i, (int)e});
      for (dlong e = 0; e < m.Nelements; e += gepb) gitems[cls].push_back({i, (int)e});
    }
    G->nitems = (int)items[cls].size() - G->item0;
    std::vector<double> eo;
    if (int st = box_even_odd_table(*any, eo)) return st;
    tab.insert(tab.end(), any->gllz.begin(), any->gllz.end());
    tab.insert(tab.end(), any->gllw.begin(), any->gllw.end());
    tab.insert(tab.end(), eo.begin(), eo.end());
  }
  if (int st = o_boxGeo.upload(geo, s)) return st;
  if (int st = o_boxTab.upload(tab, s)) return st;
  for (int cls = 0; cls < 2; ++cls) {
    if (int st = boxItems[cls].upload(items[cls], s)) return st;
    if (int st = gatherItems[cls].upload(gitems[cls], s)) return st;
  }

  // ---- concatenated gather maps, super-blocks and chunks
  std::vector<dlong> rowStarts(1, 0), colIds;
  std::vector<BatchSuper> supers;
  std::vector<BatchChunk> chunks;
  std::vector<int2> pApRange(nprob), rrRange(nprob);
  colIds.reserve(NLocalTot);
  for (int i = 0; i < nprob; ++i) {
    const ogs::ogs_t& o = ogss[i];
    const dlong nnz0 = (dlong)colIds.size();
    for (dlong r = 0; r < o.Ngather; ++r) rowStarts.push_back(nnz0 + o.rowStartsT[r + 1]);
    for (dlong g = 0; g < o.nnzT; ++g) colIds.push_back((dlong)(localOff[i] + o.colIdsT[g]));
    pApRange[i].x = (int)supers.size();
    for (dlong b = 0; b < o.NrowBlocksT; b += kSuperBlocks) {
      const dlong b1 = std::min<dlong>(b + kSuperBlocks, o.NrowBlocksT);
      supers.push_back({i, off[i] + o.blockRowStartsT[b], off[i] + o.blockRowStartsT[b1], 0});
    }
    pApRange[i].y = (int)supers.size();
    rrRange[i].x = (int)chunks.size();
    const dlong n = o.Ngather;
    if (n == 0) chunks.push_back({i, off[i], off[i], 0});  // still initialises the state
    for (dlong c = 0; c < n; c += kChunk)
      chunks.push_back({i, off[i] + c, off[i] + std::min<dlong>(c + kChunk, n), c / kChunk});
    rrRange[i].y = (int)chunks.size();
  }
  // r.r partials of the FP64 solve: per problem room for the chunks' of the
  // initial residual and the gather workgroups' of the later ones
  int nrr = 0;
  for (int i = 0; i < nprob; ++i) {
    BoxBatchProb& pr = probs[i];
    const int epb = box_gather_elements(meshes[i].Nq);
    pr.rr0 = nrr;
    pr.ninit = rrRange[i].y - rrRange[i].x;
    pr.nrr = (meshes[i].Nelements + epb - 1) / epb;
    nrr += std::max(pr.ninit, pr.nrr);
  }
  if (int st = o_probs.upload(probs, s)) return st;
  nsupers = (int)supers.size();
  nchunks = (int)chunks.size();
  if (int st = o_rowStarts.upload(rowStarts, s)) return st;
  if (int st = o_colIds.upload(colIds, s)) return st;
  if (int st = o_supers.upload(supers, s)) return st;
  if (int st = o_chunks.upload(chunks, s)) return st;
  if (int st = o_pApRange.upload(pApRange, s)) return st;
  if (int st = o_rrRange.upload(rrRange, s)) return st;
  if (int st = o_state.alloc(nprob)) return st;
  if (int st = o_r.alloc(std::max<dlong>(Ntot, 1))) return st;
  if (int st = o_p.alloc(std::max<dlong>(Ntot, 1))) return st;
  if (int st = o_Ap.alloc(std::max<dlong>(Ntot, 1))) return st;
  if (int st = o_AqL.alloc(std::max<dlong>(NLocalTot, 1))) return st;
  if (int st = o_x.alloc(std::max<dlong>(Ntot, 1))) return st;
  if (int st = o_part_rr.alloc(std::max({nchunks, nrr, 1}))) return st;
  if (int st = o_part_pAp.alloc(std::max({nsupers, npAp, 1}))) return st;
  if (int st = o_count.alloc(1)) return st;
  BPX_HIP(hipMemsetAsync(o_state.ptr(), 0, sizeof(BatchState) * nprob, s));
  BPX_HIP(hipMemsetAsync(o_p.ptr(), 0, sizeof(double) * std::max<dlong>(Ntot, 1), s));
  BPX_HIP(hipStreamSynchronize(s));
  return Tune();
}

// the Ax of the problems that their states do not skip
BoxAxArgs<double> bp_batch_t::BoxArgs(int cls, const double* q, int item0, int nitems) {
  BoxAxArgs<double> a;
  a.geo = o_boxGeo.ptr();
  a.tab = o_boxTab.ptr();
  a.lambda = lambda;
  a.q = q;
  a.AqL = o_AqL.ptr();
  a.nitems = nitems < 0 ? (int)boxItems[cls].length() : nitems;
  a.items = boxItems[cls].ptr() + item0;
  a.probs = o_probs.ptr();
  a.bst = o_state.ptr();
  return a;
}

// Times each degree's Ax (the box kernel has one workgroup shape)
int bp_batch_t::Tune() {
  hipEvent_t t0, t1;
  BPX_HIP(hipEventCreate(&t0));
  if (hipEventCreate(&t1) != hipSuccess) {
    (void)hipEventDestroy(t0);
    return set_error(BPX_ERR_HIP, "batch tune: event create failed");
  }
  int st = BPX_OK;
  for (auto& G : groups) {
    const int cls = box_batch_class(G.N);
    const BoxAxArgs<double> a = BoxArgs(cls, o_p.ptr(), G.item0, G.nitems);
    if ((st = launch_box_batch_ax(stream, cls, a))) break;  // warm-up
    float ms = 0;
    if (hipEventRecord(t0, stream) != hipSuccess || (st = launch_box_batch_ax(stream, cls, a)) ||
        hipEventRecord(t1, stream) != hipSuccess || hipEventSynchronize(t1) != hipSuccess ||
        hipEventElapsedTime(&ms, t0, t1) != hipSuccess) {
      if (!st) st = set_error(BPX_ERR_HIP, "batch tune: event timing failed");
      break;
    }
    G.us = ms * 1e3;
  }
  (void)hipEventDestroy(t0);
  (void)hipEventDestroy(t1);
  return st;
}

// One CG iteration of the problems still running
int bp_batch_t::Iteration() {
  for (int cls = 0; cls < 2; ++cls) {
    BoxAxArgs<double> a = BoxArgs(cls, o_p.ptr());
    a.fold = 1;
    a.p = o_Ap.ptr();  // the second direction (Ap itself is never stored)
    a.r = o_r.ptr();
    a.x = o_x.ptr();
    a.part = o_part_pAp.ptr();
    a.part_rr = o_part_rr.ptr();
    if (int st = launch_box_batch_ax(stream, cls, a)) return st;
    BoxBatchUpdate u;
    u.nitems = (int)gatherItems[cls].length();
    u.items = gatherItems[cls].ptr();
    u.probs = o_probs.ptr();
    u.st = o_state.ptr();
    u.AqL = o_AqL.ptr();
    u.r = o_r.ptr();
    u.part_pAp = o_part_pAp.ptr();
    u.part_rr = o_part_rr.ptr();
    if (int st = launch_box_batch_update_r(stream, cls, u)) return st;
  }
  return BPX_OK;
}

// kGraphIters iterations and the count of finished problems. The solution
// and the tolerance are the batch's own memory, so one graph serves every
// call.
int bp_batch_t::Capture() {
  if (graphExec) return BPX_OK;
  BPX_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
  int st = BPX_OK;
  for (int k = 0; k < kGraphIters && st == BPX_OK; ++k) st = Iteration();
  if (st == BPX_OK) st = launch_batch_count_done(stream, nprob, o_state.ptr(), o_count.ptr());
  hipGraph_t graph = nullptr;
  const hipError_t e = hipStreamEndCapture(stream, &graph);
  if (st) {
    if (graph) (void)hipGraphDestroy(graph);
    return st;
  }
  if (e != hipSuccess) return hip_error(e, "hipStreamEndCapture");
  const hipError_t e2 = hipGraphInstantiate(&graphExec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e2 != hipSuccess) {
    graphExec = nullptr;
    return hip_error(e2, "hipGraphInstantiate");
  }
  return BPX_OK;
}

int bp_batch_t::Solve(double* o_x, const double* o_b, double tol, int maxit, int* iterations, double* rnorm,
                      int* breakdown) {
  if (maxit < 0) return set_error(BPX_ERR_INVALID_ARGUMENT, "batch: maxit < 0");
  if (Ntot > 0 && (!o_x || !o_b)) return set_error(BPX_ERR_INVALID_ARGUMENT, "batch: null vector");
  // order after the caller's work on the platform stream
  BPX_HIP(hipEventRecord(ev0, platform->stream));
  BPX_HIP(hipStreamWaitEvent(stream, ev0, 0));
  if (int st = launch_batch_init(stream, nchunks, o_chunks.ptr(), o_b, this->o_x.ptr(), o_r.ptr(), o_probs.ptr(),
                                 o_part_rr.ptr(), o_state.ptr(), tol, maxit))
    return st;
  if (int st = Capture()) return st;
  // every replay runs kGraphIters iterations of the problems still going;
  // maxit/kGraphIters + 1 replays let the last one reach its cap and stop
  const long long maxReplays = (long long)maxit / kGraphIters + 2;
  replays = 0;
  // the count of replay rep is read while replay rep + 1 runs (a replay past
  // the end finds every problem done and does nothing); both entries of
  // h_count are the stream's until the wait below
  for (long long rep = 0; rep < maxReplays; ++rep) {
    BPX_HIP(hipGraphLaunch(graphExec, stream));
    BPX_HIP(hipMemcpyAsync(h_count + (rep & 1), o_count.ptr(), sizeof(int), hipMemcpyDeviceToHost, stream));
    BPX_HIP(hipEventRecord(evCount[rep & 1], stream));
    ++replays;
    if (rep == 0) continue;
    BPX_HIP(hipEventSynchronize(evCount[(rep - 1) & 1]));
    if (h_count[(rep - 1) & 1] >= nprob) break;
  }
  if (Ntot > 0)
    BPX_HIP(hipMemcpyAsync(o_x, this->o_x.ptr(), (size_t)Ntot * sizeof(double), hipMemcpyDeviceToDevice, stream));
  std::vector<BatchState> hs(nprob);
  BPX_HIP(hipMemcpyAsync(hs.data(), o_state.ptr(), sizeof(BatchState) * nprob, hipMemcpyDeviceToHost, stream));
  // x and the states are complete on return: the stream is the batch's own,
  // which neither the caller nor the null stream waits for
  BPX_HIP(hipStreamSynchronize(stream));
  int anyBreak = 0;
  for (int i = 0; i < nprob; ++i) {
    if (iterations) iterations[i] = hs[i].iter;
    if (rnorm) rnorm[i] = hs[i].rnorm;
    if (breakdown) breakdown[i] = hs[i].breakdown;
    anyBreak |= hs[i].breakdown;
  }
  BPX_HIP(hipEventRecord(ev1, stream));
  BPX_HIP(hipStreamWaitEvent(platform->stream, ev1, 0));
  if (anyBreak) return set_error(BPX_ERR_BREAKDOWN, "batch: CG breakdown in at least one problem");
  return BPX_OK;
}

// ---- FP32 CG with FP64 corrections, every problem at once -------------
// The recurrence of bp_t::SolveMixed per problem: FP32 vectors and
// operator (factors rounded to FP32), FP64 dot products, and every
// `interval` iterations x += c and r = float(b - A x) with the FP64
// operator, where the stopping test is made. Problems advance in lockstep
// segments (interval FP32 iterations, then the correction), captured once
// as a hipGraph; a finished problem's elements, rows and chunks return at
// once in every kernel of later segments.

int bp_batch_t::Prepare32() {
  if (have32) return BPX_OK;
  hipStream_t s = stream;
  for (auto& G : groups) {
    int st;
    if ((st = G.wJ32.alloc(G.wJ.length())) || (st = G.ggeo32.alloc(G.ggeo.length())) ||
        (st = G.D32.alloc(G.D.length())))
      return st;
    if ((st = launch_to_f32(s, G.wJ.length(), G.wJ.ptr(), G.wJ32.ptr())) ||
        (st = launch_to_f32(s, G.ggeo.length(), G.ggeo.ptr(), G.ggeo32.ptr())) ||
        (st = launch_to_f32(s, G.D.length(), G.D.ptr(), G.D32.ptr())))
      return st;
  }
  const size_t n = std::max<dlong>(Ntot, 1), nl = std::max<dlong>(NLocalTot, 1);
  int st;
  if ((st = o_r32.alloc(n)) || (st = o_p32.alloc(n)) || (st = o_Ap32.alloc(n)) || (st = o_c32.alloc(n)) ||
      (st = o_AqL32.alloc(nl)) || (st = o_Ax64.alloc(n)) || (st = o_part_true.alloc(std::max(nchunks, 1))) ||
      (st = o_inner.alloc(nprob)))
    return st;
  BPX_HIP(hipStreamSynchronize(s));
  have32 = true;
  return BPX_OK;
}

// interval FP32 iterations, then the FP64 correction and the stopping test
int bp_batch_t::Segment(double* o_x, const double* o_b, double tol, int interval) {
  BatchState* in = o_inner.ptr();
  BatchState* out = o_state.ptr();
  const float lam32 = (float)lambda;
  for (int j = 0; j < interval; ++j) {
    if (int st = launch_bm_update_p(stream, nchunks, o_chunks.ptr(), o_rrRange.ptr(), o_r32.ptr(), o_p32.ptr(),
                                    o_part_rr.ptr(), in, out))
      return st;
    for (const auto& G : groups)
      if (int st = launch_bp5_batch_f32(stream, G.N, (int)G.Nel, G.elementList.ptr(), G.G2L.ptr(), G.wJ32.ptr(),
                                        G.ggeo32.ptr(), G.D32.ptr(), lam32, o_p32.ptr(), o_AqL32.ptr() + G.loff,
                                        G.elemPid.ptr(), in))
        return st;
    if (int st = launch_batch_gather_f32(stream, nsupers, o_supers.ptr(), o_rowStarts.ptr(), o_colIds.ptr(),
                                         o_AqL32.ptr(), o_Ap32.ptr(), o_p32.ptr(), o_part_pAp.ptr(), in))
      return st;
    if (int st = launch_bm_update_xr(stream, nchunks, o_chunks.ptr(), o_pApRange.ptr(), o_p32.ptr(), o_Ap32.ptr(),
                                     o_c32.ptr(), o_r32.ptr(), o_part_pAp.ptr(), o_part_rr.ptr(), in, out))
      return st;
  }
  if (int st = launch_bm_flush(stream, nchunks, o_chunks.ptr(), o_c32.ptr(), o_x, out)) return st;
  for (int cls = 0; cls < 2; ++cls)  // (the outer states are o_state)
    if (int st = launch_box_batch_ax(stream, cls, BoxArgs(cls, o_x))) return st;
  if (int st = launch_batch_gather_only(stream, nsupers, o_supers.ptr(), o_rowStarts.ptr(), o_colIds.ptr(),
                                        o_AqL.ptr(), o_Ax64.ptr(), out))
    return st;
  if (int st = launch_bm_true_residual(stream, nchunks, o_chunks.ptr(), o_b, o_Ax64.ptr(), o_r32.ptr(),
                                       o_part_true.ptr(), o_part_rr.ptr(), out))
    return st;
  if (int st = launch_bm_decide(stream, nprob, o_rrRange.ptr(), o_part_true.ptr(), in, out, tol, 0)) return st;
  return launch_batch_count_done(stream, nprob, out, o_count.ptr());
}

int bp_batch_t::CaptureMixed(double* o_x, const double* o_b, double tol, int interval) {
  if (graphMixed && graphMixedX == o_x && graphMixedB == o_b && graphMixedTol == tol &&
      graphMixedInterval == interval)
    return BPX_OK;
  if (graphMixed) {
    (void)hipGraphExecDestroy(graphMixed);
    graphMixed = nullptr;
  }
  BPX_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
  const int st = Segment(o_x, o_b, tol, interval);
  hipGraph_t graph = nullptr;
  const hipError_t e = hipStreamEndCapture(stream, &graph);
  if (st) {
    if (graph) (void)hipGraphDestroy(graph);
    return st;
  }
  if (e != hipSuccess) return hip_error(e, "hipStreamEndCapture");
  const hipError_t e2 = hipGraphInstantiate(&graphMixed, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e2 != hipSuccess) {
    graphMixed = nullptr;
    return hip_error(e2, "hipGraphInstantiate");
  }
  graphMixedX = o_x;
  graphMixedB = o_b;
  graphMixedTol = tol;
  graphMixedInterval = interval;
  return BPX_OK;
}

int bp_batch_t::SolveMixed(double* o_x, const double* o_b, double tol, int interval, int maxit, int* iterations,
                           int* updates, double* relres, int* breakdown) {
  if (!(tol > 0) || interval < 1 || maxit < 1)
    return set_error(BPX_ERR_INVALID_ARGUMENT, "batch mixed solve: tol > 0, interval >= 1 and maxit >= 1 required");
  if (Ntot > 0 && (!o_x || !o_b)) return set_error(BPX_ERR_INVALID_ARGUMENT, "batch: null vector");
  if (int st = Prepare32()) return st;
  BPX_HIP(hipEventRecord(ev0, platform->stream));
  BPX_HIP(hipStreamWaitEvent(stream, ev0, 0));
  BatchState* in = o_inner.ptr();
  BatchState* out = o_state.ptr();
  if (int st = launch_bm_init(stream, nchunks, o_chunks.ptr(), o_b, o_x, o_r32.ptr(), o_c32.ptr(),
                              o_part_true.ptr(), o_part_rr.ptr(), in, out, maxit))
    return st;
  if (int st = launch_bm_decide(stream, nprob, o_rrRange.ptr(), o_part_true.ptr(), in, out, tol, 1)) return st;
  if (int st = CaptureMixed(o_x, o_b, tol, interval)) return st;
  // a segment adds up to `interval` FP32 iterations per running problem;
  // once a problem reaches maxit its recurrence pauses and the next
  // correction ends it
  const long long maxReplays = (long long)maxit / interval + 2;
  replays = 0;
  for (long long rep = 0; rep < maxReplays; ++rep) {
    BPX_HIP(hipGraphLaunch(graphMixed, stream));
    BPX_HIP(hipMemcpyAsync(h_count, o_count.ptr(), sizeof(int), hipMemcpyDeviceToHost, stream));
    BPX_HIP(hipStreamSynchronize(stream));
    ++replays;
    if (*h_count >= nprob) break;
  }
  std::vector<BatchState> ho(nprob), hi(nprob);
  BPX_HIP(hipMemcpy(ho.data(), out, sizeof(BatchState) * nprob, hipMemcpyDeviceToHost));
  BPX_HIP(hipMemcpy(hi.data(), in, sizeof(BatchState) * nprob, hipMemcpyDeviceToHost));
  int anyBreak = 0;
  for (int i = 0; i < nprob; ++i) {
    if (iterations) iterations[i] = ho[i].iter;
    if (updates) updates[i] = ho[i].updates;
    if (relres) relres[i] = hi[i].tol2 > 0 ? ho[i].rnorm / std::sqrt(hi[i].tol2) : 0.0;
    if (breakdown) breakdown[i] = ho[i].breakdown;
    anyBreak |= ho[i].breakdown;
  }
  BPX_HIP(hipEventRecord(ev1, stream));
  BPX_HIP(hipStreamWaitEvent(platform->stream, ev1, 0));
  if (anyBreak) return set_error(BPX_ERR_BREAKDOWN, "batch mixed solve: non-finite residual in at least one problem");
  return BPX_OK;
}

}  // namespace bpx
