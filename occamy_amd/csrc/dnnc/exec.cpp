// Executor: walks a compiled DNN program and issues one runtime call per
// operation, which is what the reference's DNN-to-LLVM lowering turns the
// program into (src/Conversion/DNNToLLVM/Ops/** build the dims arrays, pass
// raw device pointers and call the row of DNNAPISpecs.inc).  The runtime is
// bound at run time from a shared object that exports include/dnnrt.h.
//
// Two ways of running a program:
//   occamy   - the reference's semantics per inference: create the pool,
//              upload every constant into its pool slot, run, copy results
//              back, wait, release the pool
//              (src/Transform/DNN/mallocPoolOpt.hpp:239-265,
//               src/Conversion/ONNXToDNN/Ops/Constant.cpp:86-90).
//   resident - the pool and a second arena holding all constants are created
//              once; an inference is input copy + kernels + output copy, and
//              the kernels can be replayed from a captured graph.
#include "exec.h"

#include <dlfcn.h>

#include <algorithm>
#include <cstring>

namespace dnnc {

#define LOAD(name)                                                            \
  do {                                                                         \
    *(void **)(&rt.name) = dlsym(rt.dl, #name);                                \
    if (!rt.name) { err = std::string("runtime library lacks ") + #name; return false; } \
  } while (0)

bool load_runtime(const std::string &path, RuntimeApi &rt, std::string &err) {
  rt.dl = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  if (!rt.dl) { err = std::string("cannot load runtime library: ") + dlerror(); return false; }
  LOAD(dnnrtCreate); LOAD(dnnrtDestroy); LOAD(dnnrtDeviceMemoryStats); LOAD(dnnrtStreamCreate); LOAD(dnnrtStreamDestroy);
  LOAD(dnnrtSetStream); LOAD(dnnrtSetTensorFormat); LOAD(dnnrtSetFilterLayout); LOAD(dnnrtSetActivationCoef); LOAD(dnnrtSetConvTile); LOAD(dnnrtListConvTiles); LOAD(dnnrtMemFill); LOAD(dnnrtMatmulNdBias); LOAD(dnnrtAttention); LOAD(dnnrtSync); LOAD(dnnrtLastError);
  LOAD(dnnrtIsHostBackend); LOAD(dnnrtGraphBegin); LOAD(dnnrtGraphEnd); LOAD(dnnrtGraphLaunch);
  LOAD(dnnrtGraphDestroy); LOAD(dnnrtEventCreate); LOAD(dnnrtEventRecord); LOAD(dnnrtEventElapsedMs);
  LOAD(dnnrtEventDestroy); LOAD(dnnrtMemPoolInit); LOAD(dnnrtMemOffset); LOAD(dnnrtMemcpy);
  LOAD(dnnrtMalloc); LOAD(dnnrtDealloc); LOAD(dnnrtHostAlloc); LOAD(dnnrtHostFree);
  LOAD(dnnrtConv); LOAD(dnnrtConvBiasActiv); LOAD(dnnrtConvBiasAddActiv); LOAD(dnnrtConvBiasActivMaxPool); LOAD(dnnrtConvBiasAddConvBiasActiv); LOAD(dnnrtActive); LOAD(dnnrtTensorOp); LOAD(dnnrtClip);
  LOAD(dnnrtErf); LOAD(dnnrtNegative); LOAD(dnnrtReciprocal); LOAD(dnnrtPow); LOAD(dnnrtCastI64toFloat);
  LOAD(dnnrtGelu); LOAD(dnnrtReduce); LOAD(dnnrtSoftmax); LOAD(dnnrtLayerNorm); LOAD(dnnrtMaxPool);
  LOAD(dnnrtAveragePool); LOAD(dnnrtMatmul2d); LOAD(dnnrtMatmulNd); LOAD(dnnrtFlatten);
  LOAD(dnnrtReshape); LOAD(dnnrtTranspose); LOAD(dnnrtGather);
  LOAD(dnnrtLeakyRelu); LOAD(dnnrtPRelu); LOAD(dnnrtConcat); LOAD(dnnrtSqueeze); LOAD(dnnrtUnsqueeze); LOAD(dnnrtExpand);
  *(void **)(&rt.dnnrtExecFenceCreate) = dlsym(rt.dl, "dnnrtExecFenceCreate");
  *(void **)(&rt.dnnrtExecStreamWait) = dlsym(rt.dl, "dnnrtExecStreamWait");
  *(void **)(&rt.dnnrtExecUpload) = dlsym(rt.dl, "dnnrtExecUpload");
  *(void **)(&rt.dnnrtExecBlockApplies) = dlsym(rt.dl, "dnnrtExecBlockApplies");
  *(void **)(&rt.dnnrtExecRunBlock) = dlsym(rt.dl, "dnnrtExecRunBlock");
  *(void **)(&rt.dnnrtExecBlockFilter) = dlsym(rt.dl, "dnnrtExecBlockFilter");
  *(void **)(&rt.dnnrtExecBlockFilterF32) = dlsym(rt.dl, "dnnrtExecBlockFilterF32");
  return true;
}
#undef LOAD

static int64_t align_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

void Session::drop_graphs() {
  if (graph) rt.dnnrtGraphDestroy(graph);
  graph = nullptr;
  for (auto &g : parked_graphs) rt.dnnrtGraphDestroy(g.second);
  parked_graphs.clear();
}

Session::~Session() {
  if (!rt.dl) return;
  drop_graphs();
  if (handle) rt.dnnrtSync(handle);
  if (pool) rt.dnnrtDealloc(pool);
  if (weights) rt.dnnrtDealloc(weights);
  for (auto &kv : staged_out) rt.dnnrtDealloc(kv.second);
  for (const Upload &u : uploads) if (u.landed) rt.dnnrtEventDestroy(u.landed);
  for (auto &kv : op_done) if (kv.second) rt.dnnrtEventDestroy(kv.second);
  if (upload_host) rt.dnnrtHostFree(upload_host);
  for (auto &kv : host_const) rt.dnnrtHostFree(kv.second);
  for (void *p : host_out) rt.dnnrtHostFree(p);
  for (void *p : host_in) rt.dnnrtHostFree(p);
  if (handle) rt.dnnrtDestroy(handle);
  if (stream) rt.dnnrtStreamDestroy(stream);
  for (dnnrtStream_t s : upload_stream) if (s) rt.dnnrtStreamDestroy(s);
}

std::string Session::rt_error(const char *what) const {
  return std::string(what) + ": " + rt.dnnrtLastError();
}

// KCRS -> KRSC, element size es
static void permute_kcrs_to_krsc(const uint8_t *src, uint8_t *dst, const Shape &w, int64_t es) {
  const int64_t K = w[0], C = w[1], R = w[2], S = w[3];
  for (int64_t k = 0; k < K; k++)
    for (int64_t c = 0; c < C; c++)
      for (int64_t r = 0; r < R; r++)
        for (int64_t s = 0; s < S; s++)
          std::memcpy(dst + (((k * R + r) * S + s) * C + c) * es, src + (((k * C + c) * R + r) * S + s) * es, (size_t)es);
}

// More than half of an fp32 filter's values are zero: its convolutions get DNNRT_CONV_ALGO_DIRECT.  Minimal filtering adds the
// nine values of a channel's filter up before it multiplies; against direct sums its relative error (2-norm) is 0.70 to 0.80
// for dense filters of 256 to 1024 channels, 0.93 to 1.07 with half the values zero, 1.43 to 1.63 with nine tenths.
static bool mostly_zero(const GTensor &t) {
  const float *v = (const float *)t.data.data();
  const int64_t n = (int64_t)(t.data.size() / sizeof(float));
  return 2 * std::count(v, v + n, 0.f) > n;
}

// KCRS -> CRSK, element size es
static void permute_kcrs_to_crsk(const uint8_t *src, uint8_t *dst, const Shape &w, int64_t es) {
  const int64_t K = w[0], CRS = w[1] * w[2] * w[3];
  for (int64_t k = 0; k < K; k++)
    for (int64_t j = 0; j < CRS; j++)
      std::memcpy(dst + (j * K + k) * es, src + (k * CRS + j) * es, (size_t)es);
}

static bool is_compute(OpKind k) { return k >= OP_CONVFWD && k < OP_RETURN; }

// The operations' stream and, where constants are uploaded ahead, those of the uploads.  These three have to be on
// hardware queues of their own: on a shared one, copies wait for the kernels in front of them and kernels for copies.  HIP
// gives a process four queues, makes one at each of the first streams, and then puts each new stream on one that has the
// fewest, which can be the one that the stream before it has just made: with one or two more streams in the process a
// ResNet-50 took 2.61 or 2.75 ms instead of 2.42.  Streams that are dropped again make all four first; of three streams
// created then in a row no two are on one queue (2.41 to 2.44 ms with 0 to 5 other sessions).
bool Session::create_streams(bool uploading, std::string &err) {
  dnnrtStream_t first[4] = {nullptr, nullptr, nullptr, nullptr};
  bool ok = true;
  for (dnnrtStream_t &s : first) ok = ok && (!uploading || !rt.dnnrtStreamCreate(&s));
  ok = ok && !rt.dnnrtStreamCreate(&stream);
  for (dnnrtStream_t &s : upload_stream) ok = ok && (!uploading || !rt.dnnrtStreamCreate(&s));
  if (!ok) err = rt_error("dnnrtStreamCreate");
  for (dnnrtStream_t s : first) if (s) rt.dnnrtStreamDestroy(s);
  if (ok && rt.dnnrtSetStream(handle, stream)) { err = rt_error("dnnrtSetStream"); ok = false; }
  return ok;
}

bool Session::init(const Program *p,const std::string &runtime_path, int mode_, std::string &err) {
  prog = p;
  mode = mode_;
  if (prog->pool_bytes < 0) { err = "the program was compiled without the pool pass"; return false; }
  if (!load_runtime(runtime_path, rt, err)) return false;
  host_backend = rt.dnnrtIsHostBackend() != 0;
  if (prog->channels_last && host_backend) { err = "channels-last programs need the GPU runtime"; return false; }
  if (rt.dnnrtCreate(&handle)) { err = rt_error("dnnrtCreate"); return false; }
  if (mode == MODE_RESIDENT && !create_streams(false, err)) return false;
  ptr.assign(prog->value_store.size(), nullptr);

  // Which constants are convolution filters and nothing else.  They are
  // re-laid once, in the pinned host copy: K,R,S,C for a channels-last (fp16)
  // program, C,R,S,K for fp32 programs on the GPU runtime.
  std::map<std::string, bool> is_filter;
  std::map<const Value *, std::string> device_copy_of;  // device tensor -> the constant uploaded into it
  for (const Op *op : prog->ops) {
    if (op->kind != OP_MEMCPY || op->mode != 1) continue;
    const Value *src = op->operands[1];
    if (!src->def || src->def->kind != OP_HOST_CONST) continue;
    const std::string &name = src->def->const_name;
    bool only_filter = true, any = false;
    for (const auto &u : op->operands[0]->uses) {
      if (u.first == op) continue;
      const bool conv = u.first->kind == OP_CONVFWD || u.first->kind == OP_CONV_BIAS_ACTIV ||
                        u.first->kind == OP_CONV_BIAS_ADD_ACTIV || u.first->kind == OP_CONV_BIAS_ACTIV_MAXPOOL ||
                        u.first->kind == OP_CONV_ADD_CONV_ACTIV;
      if (conv && (u.second == 1 || (u.first->kind == OP_CONV_ADD_CONV_ACTIV && u.second == 5))) any = true;
      else if (is_compute(u.first->kind)) only_filter = false;
    }
    const bool f = any && only_filter;
    auto it = is_filter.find(name);
    if (it == is_filter.end()) is_filter[name] = f;
    else it->second = it->second && f;
    device_copy_of[op->operands[0]] = name;
  }
  // The two filters of a fused shortcut pair go to one kernel, which takes one layout: if one of them has to
  // stay as it is (another operator reads the same constant), so does the other.
  for (bool changed = true; changed;) {
    changed = false;
    for (const Op *op : prog->ops) {
      if (op->kind != OP_CONV_ADD_CONV_ACTIV) continue;
      const auto a = device_copy_of.find(op->operands[1]), b = device_copy_of.find(op->operands[5]);
      if (a == device_copy_of.end() || b == device_copy_of.end()) continue;
      bool &fa = is_filter[a->second], &fb = is_filter[b->second];
      if (fa != fb) { fa = fb = false; changed = true; }
    }
  }

  // Constants: one pinned host copy each (the reference keeps them as globals
  // of the model library); function results: one pinned buffer each.
  int64_t weight_bytes = 0;
  for (const Op *op : prog->ops) {
    if (op->kind == OP_HOST_CONST) {
      const GTensor &t = prog->graph->tensors.at(op->const_name);
      void *h = nullptr;
      if (rt.dnnrtHostAlloc(&h, (int64_t)t.data.size())) { err = rt_error("dnnrtHostAlloc"); return false; }
      const auto fit = is_filter.find(op->const_name);
      const bool filter = fit != is_filter.end() && fit->second && t.shape.size() == 4;
      if (filter && prog->channels_last) {
        permute_kcrs_to_krsc(t.data.data(), (uint8_t *)h, t.shape, dtype_bytes(t.dtype));
      } else if (filter && !host_backend && t.dtype == F32) {
        permute_kcrs_to_crsk(t.data.data(), (uint8_t *)h, t.shape, dtype_bytes(t.dtype));
        crsk_const[op->const_name] = true;
        if (t.shape[2] == 3 && t.shape[3] == 3 && mostly_zero(t)) sparse_const.insert(op->const_name);
      } else {
        std::memcpy(h, t.data.data(), t.data.size());
      }
      host_const[op->const_name] = h;
      ptr[(size_t)op->result->id] = h;
      weight_bytes += align_up((int64_t)t.data.size(), 256);
    } else if (op->kind == OP_HOST_ALLOC) {
      void *h = nullptr;
      if (rt.dnnrtHostAlloc(&h, op->bytes)) { err = rt_error("dnnrtHostAlloc"); return false; }
      if ((size_t)op->out_index >= host_out.size()) host_out.resize((size_t)op->out_index + 1, nullptr);
      host_out[(size_t)op->out_index] = h;
      ptr[(size_t)op->result->id] = h;
    }
  }
  filter_crsk.assign(prog->value_store.size(), 0);
  for (const Op *op : prog->ops) {
    if (op->kind != OP_MEMCPY || op->mode != 1) continue;
    const Value *src = op->operands[1];
    if (src->def && src->def->kind == OP_HOST_CONST && crsk_const.count(src->def->const_name))
      filter_crsk[(size_t)op->operands[0]->id] = 1;
  }
  for (const Value *a : prog->args) {
    void *h = nullptr;
    if (rt.dnnrtHostAlloc(&h, shape_numel(a->shape) * dtype_bytes(a->dtype))) { err = rt_error("dnnrtHostAlloc"); return false; }
    host_in.push_back(h);
  }
  weights_bytes = weight_bytes;

  if (mode == MODE_RESIDENT) {
    if (rt.dnnrtMemPoolInit(&pool, std::max(prog->pool_bytes, prog->pool_extent))) { err = rt_error("dnnrtMemPoolInit"); return false; }
    if (rt.dnnrtMalloc(&weights, weight_bytes)) { err = rt_error("dnnrtMalloc(weights)"); return false; }
    // Upload every constant once, into the weights arena; the pool slot the
    // planner gave it stays unused.
    int64_t woff = 0;
    for (const Op *op : prog->ops) {
      if (op->kind == OP_MEMPOOL_INIT) ptr[(size_t)op->result->id] = pool;
      else if (op->kind == OP_MEM_OFFSET) ptr[(size_t)op->result->id] = (char *)pool + op->offset;
    }
    for (const Op *op : prog->ops) {
      if (op->kind != OP_MEMCPY || op->mode != 1) continue;
      const Value *src = op->operands[1];
      if (!src->def || src->def->kind != OP_HOST_CONST) continue;
      void *dev = (char *)weights + woff;
      woff += align_up(op->bytes, 256);
      if (rt.dnnrtMemcpy(dev, ptr[(size_t)src->id], op->bytes, 1, stream)) { err = rt_error("dnnrtMemcpy(constant)"); return false; }
      ptr[(size_t)op->operands[0]->id] = dev;
    }
    if (rt.dnnrtSync(handle)) { err = rt_error("dnnrtSync"); return false; }
    // a result that is copied out before the last compute operation
    bool compute_later = false;
    for (auto it = prog->ops.rbegin(); it != prog->ops.rend(); ++it) {
      const Op *op = *it;
      if (is_compute(op->kind)) compute_later = true;
      if (op->kind != OP_MEMCPY || op->mode != 2 || !compute_later) continue;
      void *stage = nullptr;
      if (rt.dnnrtMalloc(&stage, op->bytes)) { err = rt_error("dnnrtMalloc(result staging)"); return false; }
      staged_out[op] = stage;
    }
  }
  for (const Op *op : prog->ops) {
    if (op->kind == OP_MEMCPY && op->mode == 1 && op->operands[1]->arg_index >= 0) callers.insert(op->operands[0]);
    if (op->kind == OP_MEMCPY && op->mode == 2) callers.insert(buffer_of(op->operands[1]));
  }
  if (mode == MODE_RESIDENT) plan_elided_copies();  // per inference, the longer lives would stand in the way of the uploads
  plan_blocks();
  // Both modes take the same blocks (the same bits): those that a per-inference program can have with its constants uploaded
  // ahead; in the reference's order a block's first filter is gone when the block runs.
  const bool ahead = !host_backend && rt.dnnrtExecFenceCreate && rt.dnnrtExecStreamWait && rt.dnnrtExecUpload;
  std::vector<UploadChunk> chunks;
  auto place = [&]() { return ahead && (mode == MODE_OCCAMY || !blocks.empty()) && place_constants(chunks); };
  bool placed = place();
  // The filters of a block lie in the pool at once: where that is too much, the block that takes the most goes.
  while (!placed && !blocks.empty()) {
    drop_block(tightest_block());
    place_block_results();
    placed = place();
  }
  for (const Block &b : blocks)
    for (const Op *op : {b.expand, b.project})
      if (op) block_filters[op->operands[1]] = {op->dimB[0], op->dimB[1]};
  if (mode == MODE_RESIDENT) {
    use_blocks = true;
    block_base = pool;
    for (const Op *op : prog->ops) {  // once more, in the block call's layout
      if (op->kind != OP_MEMCPY || op->mode != 1) continue;
      const auto f = block_filters.find(op->operands[0]);
      if (f == block_filters.end()) continue;
      uint8_t *host = (uint8_t *)ptr[(size_t)op->operands[1]->id];
      const std::vector<uint8_t> rows(host, host + op->bytes);
      block_filter(f->first)(host, rows.data(), f->second.first, f->second.second);
      if (rt.dnnrtMemcpy(ptr[(size_t)op->operands[0]->id], host, op->bytes, 1, stream)) { err = rt_error("dnnrtMemcpy(constant)"); return false; }
    }
    if (!block_filters.empty() && rt.dnnrtSync(handle)) { err = rt_error("dnnrtSync"); return false; }
    return true;
  }
  if (!create_streams(placed && !chunks.empty(), err)) return false;
  return !placed || plan_uploads(chunks, err);
}

static bool is_conv_call(const Op *op) { return op->kind == OP_CONV_BIAS_ACTIV || op->kind == OP_CONV_BIAS_ADD_ACTIV; }

void Session::fill_block(const Block &b, dnnrtExecBlock &k) const {
  auto P = [&](const Op *op, size_t i) { return ptr[(size_t)op->operands[i]->id]; };
  const Op *first = b.expand ? b.expand : b.dw;
  k = dnnrtExecBlock{};
  k.expand = b.expand != nullptr;
  k.x = P(first, 0);
  if (b.expand) { k.w1 = P(b.expand, 1); k.b1 = P(b.expand, 2); k.act1 = b.expand->mode; k.coef1 = b.expand->coef; }
  k.wd = P(b.dw, 1); k.bd = P(b.dw, 2); k.actd = b.dw->mode; k.coefd = b.dw->coef;
  k.w3 = P(b.project, 1); k.b3 = P(b.project, 2); k.act = b.project->mode; k.coef = b.project->coef;
  k.z = b.project->kind == OP_CONV_BIAS_ADD_ACTIV ? P(b.project, 4) : nullptr;
  k.y = b.y_off >= 0 ? (char *)block_base + b.y_off : P(b.project, b.project->operands.size() - 1);
  k.n = first->dimA[0]; k.cin = first->dimA[1]; k.h = first->dimA[2]; k.w = first->dimA[3];
  k.ch = b.dw->dimB[0]; k.r = b.dw->dimB[2]; k.s = b.dw->dimB[3]; k.stride = b.dw->strides[0]; k.pad_h = b.dw->pads[0]; k.pad_w = b.dw->pads[1];
  k.p = b.project->dimA[2]; k.q = b.project->dimA[3]; k.cout = b.project->dimB[0];
  k.dtype = (int32_t)b.project->operands.back()->dtype;
  k.format = format_for(first);
}

// The slots of everything but constants: from the first operation that uses one to the last.  A block's inner tensors
// have none, and its operands are read where its last convolution stands.
std::map<const Value *, Session::Range> Session::live_slots() const {
  std::map<const Value *, Range> live;
  std::map<const Value *, const Value *> home;  // value -> the slot it lives in
  std::map<const Value *, bool> constant;
  int n = 0;
  auto touch = [&](const Value *v, int at) {
    const auto h = home.find(v);
    if (h == home.end() || h->second->def->bytes <= 0 || constant.count(h->second)) return;
    const Value *s = h->second;
    const auto l = live.emplace(s, Range{s->def->offset, s->def->offset + s->def->bytes, at, at}).first;
    l->second.last = std::max(l->second.last, at);
  };
  for (const Op *op : prog->ops) {
    if (op->kind == OP_MEM_OFFSET) {
      home[op->result] = op->result;
    } else if (op->kind == OP_MEMCPY && op->mode == 1) {
      const Value *src = op->operands[1];
      if (src->def && src->def->kind == OP_HOST_CONST) constant[op->operands[0]] = true;
      else touch(op->operands[0], 0);  // an argument: from the start
    } else if (op->kind == OP_MEMCPY) {
      for (const Value *v : op->operands) touch(v, n);
    } else if (is_compute(op->kind)) {
      if (elided.count(op)) {  // its result lives on in its input's slot
        touch(op->operands[0], n);
        const auto h = home.find(op->operands[0]);
        if (h != home.end()) home[op->result] = h->second;
        n++;
        continue;
      }
      const auto b = block_of.find(op);
      const int at = b == block_of.end() ? n : blocks[(size_t)b->second].at;
      const bool inner = b != block_of.end() && op != blocks[(size_t)b->second].project;
      for (size_t i = 0; i < op->operands.size(); i++)
        if (!inner || i + 1 < op->operands.size()) touch(op->operands[i], at);
      if (!inner && !op->operands.empty()) {
        const auto h = home.find(op->operands.back());
        if (h != home.end()) home[op->result] = h->second;
      }
      n++;
    }
  }
  return live;
}

static bool moves_nothing(const Op *op) {
  return (op->kind == OP_FLATTEN || op->kind == OP_RESHAPE || op->kind == OP_SQUEEZE || op->kind == OP_UNSQUEEZE) && op->operands.size() == 2;
}
// The buffer is named by its writers alone (nobody reads it past the result, no copy to the host).
static bool plain_buffer(const Op *op) {
  const Value *s = op->operands.back();
  if (!s->def || s->def->kind != OP_MEM_OFFSET) return false;
  for (const auto &u : s->uses)
    if (!is_compute(u.first->kind) || u.second + 1 != (int)u.first->operands.size()) return false;
  return true;
}

// Copies that move no element need not run where their input's bytes stay as they are until the copy's last reader (the
// planner's lifetimes say so) and lie in the pool: what a run in place has at the caller's address need not be aligned as
// the copy is.  (The alias_copies pass does the same to the program; one compiled without it still has the
// calls and the slots, a launch of 4.5 us or a pass over memory each.)  SRGAN's generator at 90x117 0.779 -> 0.759 ms,
// SSD300 1.622 -> 1.609, AlexNet at batch 1 0.136 -> 0.131; what is left is overwritten by the next operation's result.
void Session::plan_elided_copies() {
  if (host_backend) return;
  std::map<const Op *, int> number;
  for (const Op *op : prog->ops)
    if (is_compute(op->kind)) { const int n = (int)number.size(); number[op] = n; }
  for (const Op *op : prog->ops) {
    if (!moves_nothing(op) || !launches(op) || !plain_buffer(op)) continue;
    bool read = true;
    for (const auto &u : op->result->uses) read = read && is_compute(u.first->kind) && u.second + 1 < (int)u.first->operands.size();
    const Value *slot = buffer_of(op->operands[0]);
    if (!read || !slot->def || slot->def->kind != OP_MEM_OFFSET || callers.count(slot)) continue;
    elided.insert(op);
    const std::map<const Value *, Range> live = live_slots();
    const auto mine = live.find(slot);
    bool ok = mine != live.end();
    for (const auto &l : live)
      if (ok && l.first != slot && l.second.lo < mine->second.hi && mine->second.lo < l.second.hi && l.second.first <= mine->second.last &&
          l.second.last >= mine->second.first)
        ok = false;
    for (const auto &u : slot->uses)  // written again
      if (is_compute(u.first->kind) && u.second + 1 == (int)u.first->operands.size() && number[u.first] > number[op]) ok = false;
    if (!ok) elided.erase(op);
  }
}

// The tensor that a value lies in: its producer's output buffer, its input's where the producer moves nothing.
const Value *Session::buffer_of(const Value *v) const {
  while (v->def && elided.count(v->def)) v = v->def->operands[0];
  return v->def && is_compute(v->def->kind) && !v->def->operands.empty() ? v->def->operands.back() : v;
}

// Which runs of two or three convolutions are one inverted residual block, and where its result goes.
//
// The planner may have put the result over the block's input (free once the expansion has read it) or, in place, over its
// residual; a kernel whose workgroups read the input while others write the result cannot have that, so the result then
// gets bytes that are free from here to its last reader: those of the two wide tensors that are not stored any more, as
// a rule.  Nothing else moves.
void Session::plan_blocks() {
  if (host_backend || !rt.dnnrtExecBlockApplies || !rt.dnnrtExecRunBlock || !rt.dnnrtExecBlockFilter || !rt.dnnrtExecBlockFilterF32) return;
  std::vector<const Op *> ops;
  std::map<const Op *, int> number;
  for (const Op *op : prog->ops)
    if (is_compute(op->kind)) { number[op] = (int)ops.size(); ops.push_back(op); }
  auto pointwise = [](const Op *op) {
    return op->group == 1 && op->dimB.size() == 4 && op->dimB[2] == 1 && op->dimB[3] == 1 && op->pads[0] == 0 && op->pads[1] == 0 && op->strides[0] == 1 && op->strides[1] == 1;
  };
  // The block call needs 16-byte aligned operands, the three calls take any.
  auto in_pool = [&](const Op *op, bool first, bool stored) {
    for (size_t i = first ? 0 : 1; i < op->operands.size() - (stored ? 0 : 1); i++)
      if (callers.count(buffer_of(op->operands[i]))) return false;
    return true;
  };
  auto only_reader = [](const Value *v, const Op *reader) { return v->uses.size() == 1 && v->uses[0].first == reader && v->uses[0].second == 0; };
  for (size_t i = 1; i < ops.size(); i++) {
    const Op *dw = ops[i - 1], *pr = ops[i];
    if (dw->kind != OP_CONV_BIAS_ACTIV || !is_conv_call(pr) || pr->operands[0] != dw->result || !pointwise(pr) || !only_reader(dw->result, pr)) continue;
    if (dw->dimB.size() != 4 || dw->group != dw->dimB[0] || dw->dimA[1] != dw->group || dw->group < 2 || dw->strides[0] != dw->strides[1]) continue;
    if (!plain_buffer(dw) || !plain_buffer(pr)) continue;
    const Op *ex = i >= 2 ? ops[i - 2] : nullptr;
    if (ex && (block_of.count(ex) || ex->kind != OP_CONV_BIAS_ACTIV || ex->result != dw->operands[0] || !pointwise(ex) || !only_reader(ex->result, dw) || !plain_buffer(ex))) ex = nullptr;
    // a filter that nothing else reads: its constant may be laid out for the block
    auto own_filter = [](const Op *op) {
      const Value *w = op->operands[1];
      if (!w->def || w->def->kind != OP_MEM_OFFSET) return false;
      int uploads_of_it = 0;
      for (const auto &u : w->uses) {
        if (u.first == op) continue;
        const Value *src = u.first->kind == OP_MEMCPY && u.first->mode == 1 && u.second == 0 ? u.first->operands[1] : nullptr;
        if (!src || !src->def || src->def->kind != OP_HOST_CONST || src->uses.size() != 1) return false;
        uploads_of_it++;
      }
      return uploads_of_it == 1;
    };
    if (!own_filter(pr) || !in_pool(pr, false, true)) continue;
    if (ex && (!own_filter(ex) || !in_pool(ex, true, false))) ex = nullptr;
    if (!in_pool(dw, !ex, false)) continue;
    bool read_later = true;  // by operations that launch something
    for (const auto &u : pr->result->uses) read_later = read_later && is_compute(u.first->kind) && launches(u.first) && !elided.count(u.first);
    if (!read_later) continue;
    // fp32 filters come C,R,S,K
    bool layouts = true;
    for (const Op *op : {ex, dw, pr}) layouts = layouts && (!op || prog->channels_last || filter_crsk[(size_t)op->operands[1]->id]);
    if (!layouts) continue;
    Block b{ex, dw, pr, (int)i, -1};
    dnnrtExecBlock k;
    fill_block(b, k);
    if (!rt.dnnrtExecBlockApplies(handle, &k)) continue;
    for (const Op *op : {ex, dw, pr})
      if (op) block_of[op] = (int)blocks.size();
    blocks.push_back(b);
  }
  place_block_results();
}

void Session::drop_block(size_t q) {
  blocks.erase(blocks.begin() + (long)q);
  block_of.clear();
  for (size_t i = 0; i < blocks.size(); i++)
    for (const Op *op : {blocks[i].expand, blocks[i].dw, blocks[i].project})
      if (op) block_of[op] = (int)i;
}

// The block during which tensors and the constants it reads take the most bytes together.
size_t Session::tightest_block() const {
  std::vector<Range> held = moved_results;
  for (const auto &l : live_slots()) held.push_back(l.second);
  size_t tightest = 0;
  int64_t most = -1;
  for (size_t q = 0; q < blocks.size(); q++) {
    int64_t bytes = 0;
    for (const Range &r : held)
      if (r.first <= blocks[q].at && r.last >= blocks[q].at) bytes += r.hi - r.lo;
    for (const Op *op : {blocks[q].expand, blocks[q].dw, blocks[q].project})
      for (size_t i = 1; op && i <= 2; i++)
        for (const auto &u : op->operands[i]->uses)
          if (u.first->kind == OP_MEMCPY && u.first->mode == 1 && u.second == 0) bytes += u.first->bytes;
    if (bytes > most) { most = bytes; tightest = q; }
  }
  return tightest;
}

// Results that would meet the block's input or residual get a place of their own.  One that cannot takes its block out,
// and as the other places rest on what is not stored, the search starts again.
void Session::place_block_results() {
  std::map<const Op *, int> number;
  for (const Op *op : prog->ops)
    if (is_compute(op->kind)) { const int n = (int)number.size(); number[op] = n; }
  for (bool again = true; again;) {
    again = false;
    moved_results.clear();
    const std::map<const Value *, Range> live = live_slots();
    std::map<const Value *, Range> moved;  // by result value
    auto bytes_of = [&](const Value *v, Range &r) -> bool {
      const auto m = moved.find(v);
      if (m != moved.end()) { r = m->second; return true; }
      const Value *s = v->def && is_compute(v->def->kind) ? v->def->operands.back() : v;
      const auto l = live.find(s);
      if (l == live.end()) return false;
      r = l->second;
      return true;
    };
    for (size_t q = 0; q < blocks.size() && !again; q++) {
      Block &b = blocks[q];
      b.y_off = -1;
      const Value *slot = b.project->operands.back();
      const int64_t size = slot->def->bytes;
      std::vector<const Value *> reads{(b.expand ? b.expand : b.dw)->operands[0]};
      if (b.project->kind == OP_CONV_BIAS_ADD_ACTIV) reads.push_back(b.project->operands[4]);
      bool meets = false, known = true;
      for (const Value *v : reads) {
        Range r;
        if (!bytes_of(v, r)) { known = false; break; }
        meets = meets || (r.lo < slot->def->offset + size && slot->def->offset < r.hi);
      }
      if (known && !meets) continue;
      int last = b.at;
      for (const auto &u : b.project->result->uses) {
        const auto o = block_of.find(u.first);
        last = std::max(last, o == block_of.end() ? number[u.first] : blocks[(size_t)o->second].at);
      }
      std::vector<Range> taken = moved_results;
      for (const auto &l : live) taken.push_back(l.second);
      std::vector<int64_t> at{0};
      for (const Range &r : taken) at.push_back(align_up(r.hi, 256));
      std::sort(at.begin(), at.end());
      for (const int64_t o : at) {
        if (!known || o + size > prog->pool_bytes) continue;
        bool ok = true;
        for (const Range &r : taken) ok = ok && !(r.lo < o + size && o < r.hi && r.first <= last && r.last >= b.at);
        if (!ok) continue;
        b.y_off = o;
        break;
      }
      if (b.y_off >= 0) {
        const Range r{b.y_off, b.y_off + size, b.at, last};
        moved_results.push_back(r);
        moved[b.project->result] = r;
      } else {
        drop_block(q);
        again = true;
      }
    }
  }
}

// Per-inference mode: where and when each constant is uploaded.
//
// Issued in program order on one stream, a constant waits for the operation in front of its reader (that operation's
// filter lies where this one goes), the reader waits for the copy, and the link idles during every kernel and the
// hand-overs between engines around it: 3.56 ms for a ResNet-50 whose 102 MB take 1.85 at the link's 55 GB/s.  The plan
// gives every constant its own place in the pool instead, the one whose bytes come free earliest on the whole, and
// streams of their own copy them in program order, each part as soon as the operations that used its bytes are done.  The
// pool stays the planned one to the byte, activations stay where the planner put them, and every constant still crosses
// the link in every inference.  Small constants that follow each other travel together (a copy costs 3.5 us beside its
// bytes, a wait of one stream for the other 15); the first chunks are small so that the first operations start early.
// (128 KB, 1.5 MB: within 2 %.)  ResNet-50 3.51 -> 2.56 ms, of which the link 1.85; MobileNetV2 1.52 -> 0.87.
// The chunks go to two streams in turn: on one stream the link idles from the last bytes of a copy over its completion and
// the event behind it to the first bytes of the next, some 5 us at each of ResNet-50's 80 copies; now the next one is under
// way, and a part whose bytes are in use holds back only every other chunk.  2.59 -> 2.42 ms, MobileNetV2 0.95 -> 0.82.
// (Parts of 512 KB: 1 % more; chunks of 2 MB: as now.)
static constexpr int64_t UPLOAD_PART_BYTES = 1 << 20;
bool Session::place_constants(std::vector<UploadChunk> &chunks) const {
  std::vector<UploadItem> items;
  std::map<const Value *, size_t> item_of;
  int n = 0;
  for (const Op *op : prog->ops) {
    if (op->kind == OP_MEMCPY && op->mode == 1) {
      const Value *src = op->operands[1], *dst = op->operands[0];
      if (!src->def || src->def->kind != OP_HOST_CONST || op->bytes <= 0) continue;
      if (item_of.count(dst)) return false;  // uploaded twice into one slot: not planned
      item_of[dst] = items.size();
      items.push_back({op, op->bytes, -1, n});
    } else if (is_compute(op->kind)) {
      const auto b = block_of.find(op);
      const int at = b == block_of.end() ? n : blocks[(size_t)b->second].at;
      for (const Value *v : op->operands) {
        const auto it = item_of.find(v);
        if (it == item_of.end()) continue;
        UploadItem &c = items[it->second];
        if (c.first < 0) c.first = at;
        c.last = std::max(c.last, at);
      }
      // A copy that is not made (the alias_copies pass) names the constant's own bytes as its result: they are read
      // until the result's last reader, as live_slots has it for everything but constants.
      if (op->result && !op->operands.empty()) {
        const auto it = item_of.find(op->operands.back());
        if (it != item_of.end()) item_of[op->result] = it->second;
      }
      n++;
    }
  }
  for (UploadItem &c : items)
    if (c.first < 0) c.first = c.last;  // nothing reads it
  std::stable_sort(items.begin(), items.end(), [](const UploadItem &a, const UploadItem &b) { return a.first < b.first; });
  std::vector<Range> slots = moved_results;
  for (const auto &l : live_slots()) slots.push_back(l.second);

  std::vector<Range> taken;
  // The bytes [o, o + k.bytes) for the chunk: its parts, or false if something else holds them while it is read.
  auto parts_at = [&](const UploadChunk &k, int64_t o, std::vector<UploadPart> &parts) -> bool {
    const int64_t end = o + k.bytes;
    if (end > prog->pool_bytes) return false;
    std::vector<int64_t> cut{o, end};
    std::vector<const Range *> met;
    for (const Range &r : taken)
      if (r.lo < end && o < r.hi && r.first <= k.last) {
        if (r.last >= k.first) return false;
        met.push_back(&r);
        cut.push_back(std::max(o, r.lo));
        cut.push_back(std::min(end, align_up(r.hi, 16)));
      }
    std::sort(cut.begin(), cut.end());
    parts.clear();
    for (size_t i = 0; i + 1 < cut.size(); i++) {
      if (cut[i] == cut[i + 1]) continue;
      int after = 0;
      for (const Range *r : met)
        if (r->lo < cut[i + 1] && cut[i] < r->hi) after = std::max(after, r->last + 1);
      if (!parts.empty() && parts.back().after == after) parts.back().hi = cut[i + 1];
      else parts.push_back({cut[i], cut[i + 1], after});
    }
    return true;
  };
  auto candidates = [&](int64_t bytes) {
    std::vector<int64_t> at{0};
    for (const Range &r : taken) {
      at.push_back(align_up(r.hi, 256));
      if (r.lo >= bytes) at.push_back((r.lo - bytes) / 256 * 256);
    }
    std::sort(at.begin(), at.end());
    return at;
  };
  auto finish_parts = [&](UploadChunk &k) {  // bytes that come free a little before the rest are not worth a copy of their own
    std::map<int, int64_t> sizes;
    for (const UploadPart &q : k.parts) sizes[q.after] += q.hi - q.lo;
    for (auto it = sizes.begin(); it != sizes.end() && std::next(it) != sizes.end(); ++it) {
      if (it->second >= UPLOAD_PART_BYTES) continue;
      const int later = std::next(it)->first;
      for (UploadPart &q : k.parts)
        if (q.after == it->first) q.after = later;
      std::next(it)->second += it->second;
    }
    for (size_t i = 0; i + 1 < k.parts.size();) {
      if (k.parts[i].after == k.parts[i + 1].after) {
        k.parts[i].hi = k.parts[i + 1].hi;
        k.parts.erase(k.parts.begin() + (long)i + 1);
      } else {
        i++;
      }
    }
    std::stable_sort(k.parts.begin(), k.parts.end(), [](const UploadPart &a, const UploadPart &b) { return a.after < b.after; });
  };
  auto chunk_of = [&](size_t lo, size_t hi) {
    UploadChunk k{{items.begin() + (long)lo, items.begin() + (long)hi}, 0, 0, items[lo].first, 0, {}};
    for (size_t i = lo; i < hi; i++) {
      k.bytes += i + 1 < hi ? align_up(items[i].bytes, 256) : items[i].bytes;
      k.last = std::max(k.last, items[i].last);
    }
    return k;
  };
  auto place_early = [&](UploadChunk &k) -> bool {
    bool found = false;
    int64_t best = 0;
    std::vector<UploadPart> parts;
    for (const int64_t o : candidates(k.bytes)) {
      if (!parts_at(k, o, parts)) continue;
      int64_t cost = 0;
      for (const UploadPart &q : parts) cost += q.after * (q.hi - q.lo);
      if (!found || cost < best) { found = true; best = cost; k.off = o; k.parts = parts; }
    }
    if (!found) return false;
    finish_parts(k);
    for (const UploadPart &q : k.parts) taken.push_back({q.lo, q.hi, q.after, k.last});
    return true;
  };
  chunks.clear();
  taken = slots;
  bool ok = true;
  int64_t target = 32 << 10;
  for (size_t i = 0; ok && i < items.size();) {
    size_t j = i;
    int64_t sum = 0;
    do sum += items[j++].bytes;
    while (j < items.size() && (sum + items[j].bytes <= target || items[j].bytes <= 8192));
    UploadChunk k = chunk_of(i, j);
    if (place_early(k)) {
      chunks.push_back(k);
    } else {
      for (size_t q = i; ok && q < j; q++) {
        UploadChunk one = chunk_of(q, q + 1);
        ok = place_early(one);
        if (ok) chunks.push_back(one);
      }
    }
    i = j;
    target = std::min<int64_t>(2 * target, 1 << 20);
  }
  if (ok) return true;
  // A pool too tight for that: each constant has its bytes only while it is read, the largest are placed first.
  chunks.clear();
  taken = slots;
  for (size_t i = 0; i < items.size(); i++) chunks.push_back(chunk_of(i, i + 1));
  std::vector<size_t> order(chunks.size());
  for (size_t i = 0; i < order.size(); i++) order[i] = i;
  std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return chunks[a].bytes > chunks[b].bytes; });
  for (const size_t i : order) {
    UploadChunk &k = chunks[i];
    bool found = false;
    for (const int64_t o : candidates(k.bytes)) {
      if (!parts_at(k, o, k.parts)) continue;
      k.off = o;
      found = true;
      break;
    }
    if (!found) return false;
    taken.push_back({k.off, k.off + k.bytes, k.first, k.last});
  }
  for (UploadChunk &k : chunks) {  // what was placed since counts too
    for (Range &r : taken)
      if (r.lo == k.off && r.hi == k.off + k.bytes && r.first == k.first && r.last == k.last) { std::swap(r, taken.back()); break; }
    const Range mine = taken.back();
    taken.pop_back();
    if (!parts_at(k, k.off, k.parts)) return false;
    taken.push_back(mine);
    finish_parts(k);
  }
  return true;
}

bool Session::plan_uploads(const std::vector<UploadChunk> &chunks, std::string &err) {
  int64_t total = 0;
  for (const UploadChunk &k : chunks) total += align_up(k.bytes, 256);
  if (!total) return true;
  if (rt.dnnrtHostAlloc(&upload_host, total)) { err = rt_error("dnnrtHostAlloc(constants)"); return false; }
  int64_t host = 0;
  std::map<size_t, void *> moved;
  int on = 0;
  for (const UploadChunk &k : chunks) {
    int64_t in = 0;
    for (const UploadItem &item : k.items) {
      const Op *copy = item.copy;
      void *at = (char *)upload_host + host + in;
      const void *from = ptr[(size_t)copy->operands[1]->id];
      const auto f = block_filters.find(copy->operands[0]);
      if (f != block_filters.end()) block_filter(f->first)(at, from, f->second.first, f->second.second);
      else std::memcpy(at, from, (size_t)item.bytes);
      moved[(size_t)copy->operands[1]->id] = at;
      upload_slots.push_back({(size_t)copy->operands[0]->id, k.off + in});
      in += align_up(item.bytes, 256);
    }
    for (size_t i = 0; i < k.parts.size(); i++) {
      const UploadPart &q = k.parts[i];
      uploads.push_back({host + q.lo - k.off, q.lo, q.hi - q.lo, k.first, k.last, q.after, on, nullptr});
      if (i + 1 == k.parts.size() && rt.dnnrtExecFenceCreate(&uploads.back().landed)) { err = rt_error("dnnrtExecFenceCreate"); return false; }
      if (q.after > 0 && !op_done[q.after] && rt.dnnrtExecFenceCreate(&op_done[q.after])) { err = rt_error("dnnrtExecFenceCreate"); return false; }
    }
    on ^= 1;
    host += align_up(k.bytes, 256);
  }
  for (const auto &m : moved) ptr[m.first] = m.second;
  for (auto it = host_const.begin(); it != host_const.end();) {  // the copies that are in use are the chunks' now
    bool used = false;
    for (const Op *op : prog->ops)
      if (op->kind == OP_HOST_CONST && ptr[(size_t)op->result->id] == it->second) used = true;
    if (used) { ++it; continue; }
    rt.dnnrtHostFree(it->second);
    it = host_const.erase(it);
  }
  return true;
}

int Session::format_for(const Op *op) const {
  if (!prog->channels_last) return 0;  // NCHW
  if (op->kind == OP_CONVFWD || op->kind == OP_CONV_BIAS_ACTIV || op->kind == OP_CONV_BIAS_ADD_ACTIV || op->kind == OP_CONV_BIAS_ACTIV_MAXPOOL ||
      op->kind == OP_CONV_ADD_CONV_ACTIV) {
    const Value *x = op->operands[0];
    // the function argument's slot holds what the host sent: NCHW
    const bool from_arg = x->def && x->def->kind == OP_MEM_OFFSET;
    return from_arg ? 2 : 1;
  }
  return 1;
}

// One compute operation -> one runtime call.
bool Session::issue(const Op *op, std::string &err) {
  if (use_blocks) {
    if (elided.count(op)) {
      ptr[(size_t)op->result->id] = ptr[(size_t)op->operands[0]->id];
      return true;
    }
    const auto it = block_of.find(op);
    if (it != block_of.end()) {
      const Block &b = blocks[(size_t)it->second];
      if (op != b.project) return true;
      dnnrtExecBlock k;
      fill_block(b, k);
      if (rt.dnnrtExecRunBlock(handle, &k)) { err = rt_error("dnnrtExecRunBlock"); return false; }
      ptr[(size_t)op->result->id] = k.y;
      return true;
    }
  }
  auto P = [&](size_t i) { return ptr[(size_t)op->operands[i]->id]; };
  void *out = op->operands.empty() ? nullptr : P(op->operands.size() - 1);
  const Value *ov = op->operands.empty() ? nullptr : op->operands.back();
  const int dt = ov ? (int)ov->dtype : 0;
  if (prog->channels_last || cur_format != 0) {
    const int f = format_for(op);
    if (f != cur_format) {
      if (rt.dnnrtSetTensorFormat(handle, f)) { err = rt_error("dnnrtSetTensorFormat"); return false; }
      cur_format = f;
    }
  }
  if (op->kind == OP_CONVFWD || op->kind == OP_CONV_BIAS_ACTIV || op->kind == OP_CONV_BIAS_ADD_ACTIV || op->kind == OP_CONV_BIAS_ACTIV_MAXPOOL ||
      op->kind == OP_CONV_ADD_CONV_ACTIV) {
    const int lay = filter_crsk[(size_t)op->operands[1]->id] ? DNNRT_FILTER_CRSK : DNNRT_FILTER_KCRS;
    if (op->kind == OP_CONV_ADD_CONV_ACTIV && filter_crsk[(size_t)op->operands[5]->id] != filter_crsk[(size_t)op->operands[1]->id]) {
      err = "executor: the two filters of a fused shortcut pair were uploaded in different layouts";
      return false;
    }
    if (lay != cur_filter_layout) {
      if (rt.dnnrtSetFilterLayout(handle, lay)) { err = rt_error("dnnrtSetFilterLayout"); return false; }
      cur_filter_layout = lay;
    }
    if ((op->mode == 3 || op->mode == 6) && op->kind != OP_CONVFWD && op->coef != cur_act_coef) {
      if (rt.dnnrtSetActivationCoef(handle, op->coef)) { err = rt_error("dnnrtSetActivationCoef"); return false; }
      cur_act_coef = op->coef;
    }
  }
  // a copy whose output buffer is its input's (the alias_copies pass): nothing to do
  if ((op->kind == OP_FLATTEN || op->kind == OP_RESHAPE || op->kind == OP_SQUEEZE || op->kind == OP_UNSQUEEZE) &&
      op->operands.size() == 2 && P(0) == out) {
    ptr[(size_t)op->result->id] = out;
    return true;
  }
  void *r = nullptr;
  auto pad4 =[](const Shape &s) { Shape o = s; while (o.size() < 4) o.push_back(1); return o; };
  switch (op->kind) {
    case OP_CONVFWD:
      r = rt.dnnrtConv(handle, P(0), op->dimA.data(), P(1), op->dimB.data(), P(2), 0, algo_operand(op, 0, op->algo), op->group,
                       op->pads.data(), op->strides.data(), out, dt);
      break;
    case OP_CONV_BIAS_ACTIV: {
      const int64_t dimB[4] = {1, op->dimB[0], 1, 1};
      r = rt.dnnrtConvBiasActiv(handle, P(0), op->dimA.data(), P(1), op->dimB.data(), P(2), dimB, P(3), 0, algo_operand(op, 0, 1),
                                op->group, op->pads.data(), op->strides.data(), op->mode, out, dt);
      break;
    }
    case OP_CONV_BIAS_ADD_ACTIV: {  // operands: x, w, bias, workspace, z, out
      const int64_t dimB[4] = {1, op->dimB[0], 1, 1};
      r = rt.dnnrtConvBiasAddActiv(handle, P(0), op->dimA.data(), P(1), op->dimB.data(), P(2), dimB, P(4), P(3), 0, algo_operand(op, 0, 1),
                                   op->group, op->pads.data(), op->strides.data(), op->mode, out, dt);
      break;
    }
    case OP_CONV_BIAS_ACTIV_MAXPOOL: {  // operands: x, w, bias, workspace, out
      const int64_t dimB[4] = {1, op->dimB[0], 1, 1};
      r = rt.dnnrtConvBiasActivMaxPool(handle, P(0), op->dimA.data(), P(1), op->dimB.data(), P(2), dimB, op->group, op->pads.data(),
                                       op->strides.data(), op->mode, op->kernel.data(), op->pool_pads.data(), op->pool_strides.data(),
                                       out, op->dimOut.data(), dt);
      break;
    }
    case OP_CONV_ADD_CONV_ACTIV:  // operands: x, w, bias, workspace, x2, w2, bias2, workspace2, out
      r = rt.dnnrtConvBiasAddConvBiasActiv(handle, P(0), op->dimA.data(), P(1), op->dimB.data(), P(2), op->pads.data(), op->strides.data(),
                                           P(4), op->dimA2.data(), P(5), op->dimB2.data(), P(6), op->pads2.data(), op->strides2.data(),
                                           op->mode, algo_operand(op, 0, 1), algo_operand(op, 1, 1), out, dt);
      break;
    case OP_ACTIVATION: {
      const Shape d = pad4(op->dimA);  // the lowering pads the dims to 4 with trailing ones
      if (d.size() > 4) {
        const int64_t flat[4] = {shape_numel(op->dimA), 1, 1, 1};
        r = rt.dnnrtActive(handle, P(0), flat, (int32_t)op->mode, out, dt);
      } else {
        r = rt.dnnrtActive(handle, P(0), d.data(), (int32_t)op->mode, out, dt);
      }
      break;
    }
    case OP_ADD:
    case OP_MUL: {
      const int32_t rank = (int32_t)op->dimA.size();
      r = rt.dnnrtTensorOp(handle, op->kind == OP_ADD ? 0 : 1, P(0), op->dimA.data(), rank, P(1), op->dimB.data(),
                           rank, out, op->dimA.data(), rank, op->coef, dt);
      break;
    }
    case OP_SQRT: {
      const int32_t rank = (int32_t)op->dimA.size();
      r = rt.dnnrtTensorOp(handle, 4, P(0), op->dimA.data(), rank, nullptr, op->dimA.data(), rank, out,
                           op->dimA.data(), rank, 1.f, dt);
      break;
    }
    case OP_NEGATIVE: r = rt.dnnrtNegative(handle, P(0), out, op->dimA.data(), (int64_t)op->dimA.size(), dt); break;
    case OP_RECIPROCAL: r = rt.dnnrtReciprocal(handle, P(0), out, op->dimA.data(), (int64_t)op->dimA.size(), dt); break;
    case OP_ERF: r = rt.dnnrtErf(handle, P(0), out, op->dimA.data(), (int64_t)op->dimA.size(), dt); break;
    case OP_GELU: r = rt.dnnrtGelu(handle, P(0), out, op->dimA.data(), (int64_t)op->dimA.size(), dt); break;
    case OP_POW: r = rt.dnnrtPow(handle, P(0), P(1), out, op->dimA.data(), (int64_t)op->dimA.size(), dt); break;
    case OP_CLIP: r = rt.dnnrtClip(handle, P(0), out, op->dimA.data(), op->lo, op->hi, (int64_t)op->dimA.size(), dt); break;
    case OP_LEAKYRELU:
      r = rt.dnnrtLeakyRelu(handle, P(0), out, op->dimA.data(), op->alpha, (int64_t)op->dimA.size(), dt);
      break;
    case OP_PRELU:
      r = rt.dnnrtPRelu(handle, P(0), out, op->dimA.data(), P(1), op->dimB.data(), (int64_t)op->dimA.size(), dt);
      break;
    case OP_CONCAT: {
      const size_t n_in = op->operands.size() - 1;
      const void *xs[16];
      const int64_t *ds[16];
      for (size_t i = 0; i < n_in; i++) { xs[i] = P(i); ds[i] = op->operands[i]->shape.data(); }
      r = rt.dnnrtConcat(handle, xs, ds, out, op->dimOut.data(), op->axis, (int64_t)n_in, (int32_t)op->dimOut.size(), dt);
      break;
    }
    case OP_SQUEEZE:
      r = rt.dnnrtSqueeze(handle, P(0), op->dimA.data(), (int64_t)op->dimA.size(), out, op->dimOut.data(),
                          (int64_t)op->dimOut.size(), dt);
      break;
    case OP_UNSQUEEZE:
      r = rt.dnnrtUnsqueeze(handle, P(0), op->dimA.data(), (int64_t)op->dimA.size(), out, op->dimOut.data(),
                            (int64_t)op->dimOut.size(), dt);
      break;
    case OP_EXPAND:  // operands: input, shape (device copy, not read), output
      r = rt.dnnrtExpand(handle, P(0), op->dimA.data(), (int64_t)op->dimA.size(), out, op->dimOut.data(),
                         (int64_t)op->dimOut.size(), dt);
      break;
    case OP_CAST:
      r = rt.dnnrtCastI64toFloat(handle, (const int64_t *)P(0), out, op->dimA.data(), (int64_t)op->dimA.size(), dt);
      break;
    case OP_REDUCE:
      r = rt.dnnrtReduce(handle, (int32_t)op->dimA.size(), P(0), op->dimA.data(), out, op->dimOut.data(),
                         (int32_t)op->mode, dt);
      break;
    case OP_MAXPOOL:
      r = rt.dnnrtMaxPool(handle, P(0), op->dimA.data(), out, op->dimOut.data(), op->kernel.data(), op->pads.data(),
                          op->strides.data(), dt);
      break;
    case OP_AVGPOOL:
      r = rt.dnnrtAveragePool(handle, P(0), op->dimA.data(), out, op->dimOut.data(), op->kernel.data(),
                              op->pads.data(), op->strides.data(), dt);
      break;
    case OP_SOFTMAX:
      r = rt.dnnrtSoftmax(handle, P(0), op->dimA.data(), out, op->dimA.data(), op->axis, (int64_t)op->dimA.size(), dt);
      break;
    case OP_LAYERNORM:
      r = rt.dnnrtLayerNorm(handle, P(0), op->dimA.data(), (int64_t)op->dimA.size(), P(1), P(2), op->eps, out, dt);
      break;
    case OP_FLATTEN:
      r = rt.dnnrtFlatten(handle, P(0), op->dimA.data(), out, op->dimOut.data(), (int32_t)op->axis,
                          (int64_t)op->dimA.size(), dt);
      break;
    case OP_RESHAPE: r = rt.dnnrtReshape(handle, P(0), op->dimA.data(), (int64_t)op->dimA.size(), out, dt); break;
    case OP_TRANSPOSE:
      r = rt.dnnrtTranspose(handle, P(0), op->dimA.data(), out, op->dimOut.data(), op->perm.data(),
                            (int64_t)op->dimA.size(), dt);
      break;
    case OP_GATHER:
      r = rt.dnnrtGather(handle, P(0), op->dimA.data(), (int64_t)op->dimA.size(), out, op->dimOut.data(),
                         (int64_t)op->dimOut.size(), (const int64_t *)P(1), op->dimB.data(), (int64_t)op->dimB.size(),
                         op->axis, dt);
      break;
    case OP_MATMUL2D:
      if (op->operands.size() == 4)  // a, b, c, out: C folded in by the matmul + bias fusion
        r = rt.dnnrtMatmul2d(handle, 2, P(0), op->dimA.data(), P(1), op->dimB.data(), P(2), op->kernel.data(), out,
                             op->dimOut.data(), op->alpha, op->beta, op->trans_a, op->trans_b, dt);
      else
        r = rt.dnnrtMatmul2d(handle, 2, P(0), op->dimA.data(), P(1), op->dimB.data(), out, op->dimOut.data(), out,
                             op->dimOut.data(), op->alpha, op->beta, op->trans_a, op->trans_b, dt);
      break;
    case OP_MATMULND:
      r = rt.dnnrtMatmulNd(handle, P(0), op->dimA.data(), (int32_t)op->dimA.size(), P(1), op->dimB.data(),
                           (int32_t)op->dimB.size(), out, op->dimOut.data(), (int32_t)op->dimOut.size(), dt);
      break;
    case OP_ATTENTION:  // operands: q, k, v, out
      if (op->axis) {  // one tensor holds [Q | K | V] per row
        const int64_t hidden = op->dimA[2];
        char *base = (char *)P(0);
        const int64_t es = dt == DNNRT_F16 ? 2 : 4;  // bytes per element
        r = rt.dnnrtAttention(handle, base, base + hidden * es, base + 2 * hidden * es, out, op->dimA[0], op->dimA[1], op->dimB[1],
                              op->group, hidden / op->group, 3 * hidden, op->alpha, dt);
      } else {
        r = rt.dnnrtAttention(handle, P(0), P(1), P(2), out, op->dimA[0], op->dimA[1], op->dimB[1], op->group,
                              op->dimA[2] / op->group, 0, op->alpha, dt);
      }
      break;
    case OP_MATMUL_BIAS:  // operands: a, b, bias, [residual,] out
      r = rt.dnnrtMatmulNdBias(handle, P(0), op->dimA.data(), (int32_t)op->dimA.size(), P(1), op->dimB.data(),
                               (int32_t)op->dimB.size(), P(2), op->operands.size() == 5 ? P(3) : nullptr, op->mode == 7,
                               out, op->dimOut.data(), (int32_t)op->dimOut.size(), dt);
      break;
    default: err = std::string("executor: unexpected op ") + op_name(op->kind); return false;
  }
  if (!r) { err = std::string(op_name(op->kind)) + ": " + rt.dnnrtLastError(); return false; }
  ptr[(size_t)op->result->id] = r;
  return true;
}

// debug_fill with the constants uploaded ahead: what held something until compute operation `n`, just issued, and is not
// read any more is filled, so that whoever reads it before it is written again gets the fill.  `held`: every tensor's and
// every constant's bytes.  In front of op_done, so that an upload into these bytes comes behind it.
bool Session::fill_dead(const std::vector<Range> &held, int n, void *base) const {
  for (const Range &dead : held) {
    if (dead.last != n) continue;
    int64_t lo = dead.lo;
    while (lo < dead.hi) {  // the pieces between what lives on
      int64_t hi = dead.hi, next = dead.hi;
      for (const Range &r : held) {
        if (r.first > n || r.last <= n || r.hi <= lo || r.lo >= hi) continue;
        if (r.lo <= lo) { hi = lo; next = r.hi; }
        else { hi = r.lo; next = r.lo; }
      }
      if (hi > lo && rt.dnnrtMemFill((char *)base + lo, debug_fill, hi - lo, stream)) return false;
      lo = next;
    }
  }
  return true;
}

// The per-inference sequence with the constants uploaded on two streams of their own (plan_uploads).
bool Session::run_uploading(const void *const *inputs, void *const *outputs, std::string &err) {
  void *run_pool = nullptr;
  size_t next = 0, landed = 0;  // the next upload to issue; those that the compute stream has waited for
  int n = 0, waited[2] = {0, 0};
  std::vector<Range> held;
  if (debug_fill >= 0) {
    held = moved_results;
    for (const auto &l : live_slots()) held.push_back(l.second);
    for (const Upload &u : uploads) held.push_back({u.dev_off, u.dev_off + u.bytes, u.after, u.last});
  }
  auto fail = [&](const char *what) { err = rt_error(what); return false; };
  // The uploads whose place is free when n operations are done.  In program order: one that has to wait holds back the rest.
  auto pump = [&]() -> bool {
    for (; next < uploads.size() && uploads[next].after <= n; next++) {
      const Upload &u = uploads[next];
      if (u.after > waited[u.on]) {
        waited[u.on] = u.after;
        if (rt.dnnrtExecStreamWait(upload_stream[u.on], op_done[u.after])) return fail("dnnrtExecStreamWait");
      }
      if (rt.dnnrtExecUpload((char *)run_pool + u.dev_off, (char *)upload_host + u.host_off, u.bytes, upload_stream[u.on])) return fail("dnnrtExecUpload(constants)");
      if (u.landed && rt.dnnrtEventRecord(u.landed, upload_stream[u.on])) return fail("dnnrtEventRecord");
    }
    return true;
  };
  auto one = [&](const Op *op) -> bool {
    switch (op->kind) {
      case OP_MEMPOOL_INIT:
        if (rt.dnnrtMemPoolInit(&run_pool, op->bytes)) return fail("dnnrtMemPoolInit");
        ptr[(size_t)op->result->id] = run_pool;
        block_base = run_pool;
        last_pool_bytes = op->bytes;
        if (debug_fill >= 0 && (rt.dnnrtMemFill(run_pool, debug_fill, op->bytes, stream) || rt.dnnrtSync(handle))) return fail("dnnrtMemFill");
        for (const Op *o : prog->ops)
          if (o->kind == OP_MEM_OFFSET && rt.dnnrtMemOffset(&ptr[(size_t)o->result->id], run_pool, o->offset, o->bytes)) return fail("dnnrtMemOffset");
        for (const auto &s : upload_slots) ptr[s.first] = (char *)run_pool + s.second;
        return pump();
      case OP_MEMCPY: {
        const Value *src = op->operands[1];
        if (op->mode == 1 && src->def && src->def->kind == OP_HOST_CONST) return true;
        if (op->mode == 1 && src->arg_index >= 0) {  // a piece crosses the link while the next is copied to pinned memory
          char *pinned = (char *)host_in[(size_t)src->arg_index];
          for (int64_t at = 0; at < op->bytes; at += 256 << 10) {
            const int64_t n_bytes = std::min<int64_t>(op->bytes - at, 256 << 10);
            std::memcpy(pinned + at, (const char *)inputs[(size_t)src->arg_index] + at, (size_t)n_bytes);
            if (rt.dnnrtExecUpload((char *)ptr[(size_t)op->operands[0]->id] + at, pinned + at, n_bytes, stream)) return fail("dnnrtExecUpload(input)");
          }
          return true;
        }
        if (rt.dnnrtMemcpy(ptr[(size_t)op->operands[0]->id], ptr[(size_t)src->id], op->bytes, (int32_t)op->mode, stream)) return fail("dnnrtMemcpy");
        return true;
      }
      case OP_DEALLOC:
        if (rt.dnnrtSync(handle)) return fail("dnnrtSync");
        if (rt.dnnrtDealloc(run_pool)) return fail("dnnrtDealloc");
        run_pool = nullptr;
        return true;
      case OP_MEM_OFFSET: case OP_HOST_CONST: case OP_HOST_ALLOC: case OP_RETURN: return true;
      default: break;
    }
    if (!pump()) return false;
    void *last_landed[2] = {nullptr, nullptr};
    for (; landed < uploads.size() && uploads[landed].first <= n; landed++)  // whole chunks: the last of their parts has the event
      last_landed[uploads[landed].on] = uploads[landed].landed;
    for (void *event : last_landed)
      if (event && rt.dnnrtExecStreamWait(stream, event)) return fail("dnnrtExecStreamWait");
    if (!issue(op, err)) return false;
    if (debug_fill >= 0 && !fill_dead(held, n, run_pool)) return fail("dnnrtMemFill");
    n++;
    const auto done = op_done.find(n);
    if (done != op_done.end() && rt.dnnrtEventRecord(done->second, stream)) return fail("dnnrtEventRecord");
    return true;
  };
  for (size_t i = 0; i < prog->args.size(); i++) ptr[(size_t)prog->args[i]->id] = host_in[i];
  for (const Op *op : prog->ops) {
    if (one(op)) continue;
    // All three streams have to be done with the pool before it goes: a copy that no event stands behind yet, too.
    for (dnnrtStream_t s : {upload_stream[0], upload_stream[1], stream}) {
      rt.dnnrtSetStream(handle, s);
      rt.dnnrtSync(handle);
    }
    if (run_pool) rt.dnnrtDealloc(run_pool);
    return false;
  }
  const Op *ret = prog->ops.back();
  for (size_t i = 0; i < ret->operands.size(); i++) {
    const Value *v = ret->operands[i];
    std::memcpy(outputs[i], ptr[(size_t)v->id], (size_t)(shape_numel(v->shape) * dtype_bytes(v->dtype)));
  }
  return true;
}

// The reference's per-inference sequence, call for call: where the constants are not uploaded ahead.
bool Session::run_occamy(const void *const *inputs, void *const *outputs, std::string &err) {
  use_blocks = !uploads.empty();
  if (use_blocks) return run_uploading(inputs, outputs, err);
  void *run_pool = nullptr;
  for (size_t i = 0; i < prog->args.size(); i++) {
    std::memcpy(host_in[i], inputs[i], (size_t)(shape_numel(prog->args[i]->shape) * dtype_bytes(prog->args[i]->dtype)));
    ptr[(size_t)prog->args[i]->id] = host_in[i];
  }
  bool ok = true;
  for (const Op *op : prog->ops) {
    switch (op->kind) {
      case OP_MEMPOOL_INIT:
        if (rt.dnnrtMemPoolInit(&run_pool, op->bytes)) { err = rt_error("dnnrtMemPoolInit"); ok = false; }
        ptr[(size_t)op->result->id] = block_base = run_pool;
        last_pool_bytes = op->bytes;
        if (ok && debug_fill >= 0 && rt.dnnrtMemFill(run_pool, debug_fill, op->bytes, stream)) { err = rt_error("dnnrtMemFill"); ok = false; }
        break;
      case OP_MEM_OFFSET: {
        void *q = nullptr;
        if (rt.dnnrtMemOffset(&q, ptr[(size_t)op->operands[0]->id], op->offset, op->bytes)) { err = rt_error("dnnrtMemOffset"); ok = false; }
        ptr[(size_t)op->result->id] = q;
        if (ok && debug_fill >= 0 && rt.dnnrtMemFill(q, debug_fill, op->bytes, stream)) { err = rt_error("dnnrtMemFill"); ok = false; }
        break;
      }
      case OP_MEMCPY:
        if (rt.dnnrtMemcpy(ptr[(size_t)op->operands[0]->id], ptr[(size_t)op->operands[1]->id], op->bytes, (int32_t)op->mode, stream)) {
          err = rt_error("dnnrtMemcpy"); ok = false;
        }
        break;
      case OP_DEALLOC:  // only the pool's own release survives the pool pass
        if (rt.dnnrtSync(handle)) { err = rt_error("dnnrtSync"); ok = false; }
        if (rt.dnnrtDealloc(ptr[(size_t)op->operands[0]->id])) { err = rt_error("dnnrtDealloc"); ok = false; }
        run_pool = nullptr;
        break;
      case OP_HOST_CONST: case OP_HOST_ALLOC: case OP_RETURN: break;
      default: ok = issue(op, err); break;
    }
    if (!ok) break;
  }
  if (!ok) {
    rt.dnnrtSync(handle);
    if (run_pool) rt.dnnrtDealloc(run_pool);
    return false;
  }
  const Op *ret = prog->ops.back();
  for (size_t i = 0; i < ret->operands.size(); i++) {
    const Value *v = ret->operands[i];
    std::memcpy(outputs[i], ptr[(size_t)v->id], (size_t)(shape_numel(v->shape) * dtype_bytes(v->dtype)));
  }
  return true;
}

bool Session::issue_all_compute(std::string &err) {
  for (const Op *op : prog->ops) {
    if (is_compute(op->kind)) {
      if (!issue(op, err)) return false;
    } else if (op->kind == OP_MEMCPY && op->mode == 2) {
      auto st = staged_out.find(op);
      if (st == staged_out.end()) continue;
      // a copy kernel, so that a captured graph holds it too
      const Value *v = op->operands[1];
      const int64_t n = shape_numel(v->shape);
      if (!rt.dnnrtReshape(handle, ptr[(size_t)v->id], &n, 1, st->second, (int32_t)v->dtype)) {
        err = rt_error("dnnrtReshape(result staging)");
        return false;
      }
    }
  }
  return true;
}

// Whether the session makes a runtime call for the operation: not for copies it elides, nor for a block's operations in
// front of its last one.
bool Session::issues(const Op *op) const {
  const auto b = block_of.find(op);
  return launches(op) && !elided.count(op) && (b == block_of.end() || op == blocks[(size_t)b->second].project);
}

const char *Session::launch_class(const Op *op) const { return block_of.count(op) ? "inverted_block" : op_class(op); }

bool Session::compute_op(int64_t i, int64_t &launch, const char *&work_class, double &flops, double &bytes) const {
  std::vector<const Op *> compute;
  for (const Op *op : prog->ops)
    if (launches(op)) compute.push_back(op);
  if (i < 0 || i >= (int64_t)compute.size()) return false;
  const Op *op = compute[(size_t)i];
  const auto at = block_of.find(op);
  const Block *b = at == block_of.end() ? nullptr : &blocks[(size_t)at->second];
  launch = elided.count(op) ? -1 : b ? std::find(compute.begin(), compute.end(), b->project) - compute.begin() : i;
  work_class = launch_class(op);
  flops = bytes = 0;
  if (!issues(op)) return true;
  if (!b) { op_work(op, flops, bytes); return true; }
  for (const Op *o : {b->expand, b->dw, b->project}) {
    if (!o) continue;
    double f, by;
    op_work(o, f, by);
    flops += f;
    bytes += by;
    if (o != b->project) bytes -= 2.0 * (double)shape_numel(o->result->shape) * (double)dtype_bytes(o->result->dtype);  // stays on the chip
  }
  return true;
}

// Resident inference.  `on_device` != 0: inputs/outputs are device pointers and
// the call returns without waiting (sync() does).
bool Session::run_resident(const void *const *inputs, void *const *outputs, int on_device, int use_graph, std::string &err) {
  const bool borrow = on_device == 2 && !host_backend;
  auto other_slot = [&](const Op *op) -> size_t {  // the pool tensor behind a result copy (see below)
    const Value *v = op->operands[1];
    if (v->def && v->def->kind == OP_MEM_OFFSET) return (size_t)v->id;
    return (size_t)v->def->operands.back()->id;
  };
  // The pool reuses the inputs' slots for later tensors, so every pass over
  // the kernels must be preceded by a fresh copy of the inputs.
  auto copy_inputs = [&]() -> bool {
    if (borrow) return true;
    for (const Op *op : prog->ops) {
      if (op->kind != OP_MEMCPY || op->mode != 1) continue;
      const Value *src = op->operands[1];
      if (src->arg_index < 0) continue;
      const size_t ai = (size_t)src->arg_index;
      const void *from = inputs[ai];
      if (!on_device) { std::memcpy(host_in[ai], inputs[ai], (size_t)op->bytes); from = host_in[ai]; }
      if (rt.dnnrtMemcpy(ptr[(size_t)op->operands[0]->id], const_cast<void *>(from), op->bytes, on_device ? 3 : 1, stream)) {
        err = rt_error("dnnrtMemcpy(input)"); return false;
      }
    }
    return true;
  };
  // on_device == 2: the kernels read the caller's input buffers where they are (no copy into the pool slots).  The
  // argument slots' values point at those buffers for as long as the caller keeps passing the same addresses; a
  // recorded graph holds them, so a change of address drops it.
  {
    bool moved = false;
    for (const Op *op : prog->ops) {
      if (op->kind != OP_MEMCPY || op->mode != 1 || op->operands[1]->arg_index < 0) continue;
      const size_t slot = (size_t)op->operands[0]->id;
      if (!arg_home.count(slot)) arg_home[slot] = ptr[slot];
      void *want = borrow ? const_cast<void *>(inputs[(size_t)op->operands[1]->arg_index]) : arg_home[slot];
      if (ptr[slot] != want) { ptr[slot] = want; moved = true; }
    }
    // The same for the results: the pool tensor a result is computed into (the output operand of the operation
    // that produces it) points at the caller's result buffer, so the last kernel writes there and no copy
    // follows.  Only that one tensor value moves: whatever else the planner put at the same pool offset at other
    // times stays in the pool, and a copy-type operation that would have aliased it copies instead.
    direct_out.clear();
    for (const Op *op : prog->ops) {
      if (op->kind != OP_MEMCPY || op->mode != 2 || staged_out.count(op)) continue;
      const Value *v = op->operands[1], *bv = nullptr;
      if (v->def && v->def->kind == OP_MEM_OFFSET) bv = v;
      else if (v->def && is_compute(v->def->kind) && !v->def->operands.empty()) {
        const Value *o = v->def->operands.back();
        if (o->def && o->def->kind == OP_MEM_OFFSET) bv = o;
      }
      if (!bv) continue;
      const size_t slot = (size_t)bv->id;
      // A second result out of one tensor, or a tensor that is also an argument's slot, is copied after the
      // kernels as before, from wherever the first result or the argument put the tensor for this run.
      bool shared = arg_home.count(slot) != 0;
      for (const Op *other : direct_out) shared = shared || other_slot(other) == slot;
      if (shared) continue;
      if (!out_home.count(slot)) out_home[slot] = ptr[slot];
      void *want = borrow ? outputs[(size_t)op->operands[0]->def->out_index] : out_home[slot];
      if (ptr[slot] != want) { ptr[slot] = want; moved = true; }
      if (borrow) direct_out.push_back(op);
    }
    // the addresses this run's kernels see: the key of its graph
    std::vector<void *> key;
    for (const auto &h : arg_home) key.push_back(ptr[h.first]);
    for (const auto &h : out_home) key.push_back(ptr[h.first]);
    if (moved || key != graph_key) {
      if (graph) {  // park the current one, take back the one recorded with these addresses if there is one
        parked_graphs.emplace_back(graph_key, graph);
        graph = nullptr;
        if (parked_graphs.size() > 4) { rt.dnnrtGraphDestroy(parked_graphs.front().second); parked_graphs.erase(parked_graphs.begin()); }
      }
      for (size_t i = 0; i < parked_graphs.size(); i++)
        if (parked_graphs[i].first == key) { graph = parked_graphs[i].second; parked_graphs.erase(parked_graphs.begin() + (long)i); break; }
      graph_key = key;
    }
  }
  // A graph launch costs the host about as much as half a dozen kernel launches: a program of up to three kernels
  // (the single convolution block: 19 us per pass replayed, 8 us launched directly) is issued as it is.
  int launching = 0;
  for (const Op *op : prog->ops) launching += issues(op) ? 1 : 0;
  const bool graphed = use_graph && !host_backend && launching > 3;
  if (graphed && !graph) {
    // One eager pass on real data first: it validates every call outside of
    // capture.  Then the same call sequence is recorded (nothing runs).
    if (!copy_inputs() || !issue_all_compute(err)) return false;
    if (rt.dnnrtSync(handle)) { err = rt_error("dnnrtSync"); return false; }
    if (rt.dnnrtGraphBegin(handle)) { err = rt_error("dnnrtGraphBegin"); return false; }
    const bool ok = issue_all_compute(err);
    void *g = nullptr;
    if (rt.dnnrtGraphEnd(handle, &g)) { if (ok) err = rt_error("dnnrtGraphEnd"); return false; }
    if (!ok) { rt.dnnrtGraphDestroy(g); return false; }
    graph = g;
  }
  // 1. inputs into their pool slots  2. kernels
  if (!copy_inputs()) return false;
  if (graphed) {
    if (rt.dnnrtGraphLaunch(handle, graph)) { err = rt_error("dnnrtGraphLaunch"); return false; }
  } else {
    if (!issue_all_compute(err)) return false;
  }
  // 3. outputs
  for (const Op *op : prog->ops) {
    if (op->kind != OP_MEMCPY || op->mode != 2) continue;
    if (std::find(direct_out.begin(), direct_out.end(), op) != direct_out.end()) continue;  // written in place
    const Op *ha = op->operands[0]->def;
    const size_t oi = (size_t)ha->out_index;
    void *dst = on_device ? outputs[oi] : host_out[oi];
    auto st = staged_out.find(op);
    void *src = st != staged_out.end() ? st->second : ptr[(size_t)op->operands[1]->id];
    if (rt.dnnrtMemcpy(dst, src, op->bytes, on_device ? 3 : 2, stream)) {
      err = rt_error("dnnrtMemcpy(output)"); return false;
    }
  }
  if (!on_device) {
    if (rt.dnnrtSync(handle)) { err = rt_error("dnnrtSync"); return false; }
    for (const Op *op : prog->ops)
      if (op->kind == OP_HOST_ALLOC) std::memcpy(outputs[(size_t)op->out_index], host_out[(size_t)op->out_index], (size_t)op->bytes);
  }
  return true;
}

bool Session::profile_resident(const void *const *inputs, int on_device, bool by_class, std::vector<float> &ms, std::string &err) {
  if (mode != MODE_RESIDENT) { err = "profiling needs a resident session"; return false; }
  // profiling copies the inputs into their pool slots: argument values that point at a caller's buffers go home
  for (const auto &h : arg_home) ptr[h.first] = h.second;
  for (const auto &h : out_home) ptr[h.first] = h.second;
  direct_out.clear();
  // the operations that launch something, in program order (an aliased copy only hands its input's address on;
  // a first eager pass has set those)
  std::vector<const Op *> compute;
  for (const Op *op : prog->ops)
    if (launches(op)) compute.push_back(op);
  for (const Op *op : prog->ops)
    if (is_compute(op->kind) && !launches(op) && !ptr[(size_t)op->result->id]) {
      std::string e2;
      if (!issue_all_compute(e2)) { err = e2; return false; }
      break;
    }
  if (by_class) return profile_classes(inputs, on_device, compute, ms, err);
  std::vector<void *> ev(compute.size() + 1, nullptr);  // [0]: the start; [i + 1]: behind operation i, if it launches in this session
  bool ok = true;
  for (size_t i = 0; ok && i < ev.size(); i++)
    if ((i == 0 || issues(compute[i - 1])) && rt.dnnrtEventCreate(&ev[i])) { err = rt_error("dnnrtEventCreate"); ok = false; }
  if (ok) {
    for (const Op *op : prog->ops) {  // inputs into their pool slots
      if (op->kind != OP_MEMCPY || op->mode != 1 || op->operands[1]->arg_index < 0) continue;
      const size_t ai = (size_t)op->operands[1]->arg_index;
      const void *from = inputs[ai];
      if (!on_device) { std::memcpy(host_in[ai], inputs[ai], (size_t)op->bytes); from = host_in[ai]; }
      if (rt.dnnrtMemcpy(ptr[(size_t)op->operands[0]->id], const_cast<void *>(from), op->bytes, on_device ? 3 : 1, stream)) {
        err = rt_error("dnnrtMemcpy(input)"); ok = false; break;
      }
    }
  }
  if (ok && rt.dnnrtEventRecord(ev[0], stream)) { err = rt_error("dnnrtEventRecord"); ok = false; }
  for (size_t i = 0; ok && i < compute.size(); i++) {
    ok = issue(compute[i], err);
    if (ok && ev[i + 1] && rt.dnnrtEventRecord(ev[i + 1], stream)) { err = rt_error("dnnrtEventRecord"); ok = false; }
  }
  if (rt.dnnrtSync(handle) && ok) { err = rt_error("dnnrtSync"); ok = false; }
  ms.assign(compute.size(), 0.f);
  for (size_t i = 0, before = 0; ok && i < compute.size(); i++) {
    if (!ev[i + 1]) continue;
    if (rt.dnnrtEventElapsedMs(ev[before], ev[i + 1], &ms[i])) { err = rt_error("dnnrtEventElapsedMs"); ok = false; }
    before = i + 1;
  }
  for (void *e : ev)
    if (e) rt.dnnrtEventDestroy(e);
  return ok;
}

// One pair of timestamps per operation class, around all of the class's
// launches issued back to back (in program order, on whatever the buffers
// hold: only the durations matter).  A timestamp between two kernels of a few
// microseconds costs about as much as the kernels; this way the class average
// is the kernels' own duration plus the gap between consecutive dispatches
// (a repeated launch finds its operands in the caches, so a small class reads
// a little faster here than inside the whole program).
bool Session::profile_classes(const void *const *inputs, int on_device, const std::vector<const Op *> &compute,
                              std::vector<float> &ms, std::string &err) {
  auto class_of = [&](const Op *op) -> std::string { return issues(op) ? launch_class(op) : ""; };
  std::vector<std::string> classes;
  for (const Op *op : compute) {
    const std::string c = class_of(op);
    if (!c.empty() && std::find(classes.begin(), classes.end(), c) == classes.end()) classes.push_back(c);
  }
  bool ok = true;
  for (const Op *op : prog->ops) {  // inputs into their pool slots
    if (op->kind != OP_MEMCPY || op->mode != 1 || op->operands[1]->arg_index < 0) continue;
    const size_t ai = (size_t)op->operands[1]->arg_index;
    const void *from = inputs[ai];
    if (!on_device) { std::memcpy(host_in[ai], inputs[ai], (size_t)op->bytes); from = host_in[ai]; }
    if (rt.dnnrtMemcpy(ptr[(size_t)op->operands[0]->id], const_cast<void *>(from), op->bytes, on_device ? 3 : 1, stream)) {
      err = rt_error("dnnrtMemcpy(input)"); return false;
    }
  }
  void *e0 = nullptr, *e1 = nullptr;
  if (rt.dnnrtEventCreate(&e0) || rt.dnnrtEventCreate(&e1)) { err = rt_error("dnnrtEventCreate"); return false; }
  ms.assign(compute.size(), 0.f);
  for (size_t i = 0; ok && i < compute.size(); i++) ok = issue(compute[i], err);  // one whole pass first: real values everywhere
  for (const std::string &c : classes) {
    if (!ok) break;
    // a class of one or two launches is repeated: behind an idle stream the first dispatch alone takes
    // longer to reach the GPU than such a kernel runs
    size_t members = 0, n = 0;
    for (const Op *op : compute) members += c == class_of(op);
    const size_t reps = members >= 32 ? 1 : (32 + members - 1) / members;
    if (rt.dnnrtEventRecord(e0, stream)) { err = rt_error("dnnrtEventRecord"); ok = false; break; }
    for (size_t r = 0; ok && r < reps; r++)
      for (size_t i = 0; ok && i < compute.size(); i++)
        if (c == class_of(compute[i])) { ok = issue(compute[i], err); n++; }
    if (ok && rt.dnnrtEventRecord(e1, stream)) { err = rt_error("dnnrtEventRecord"); ok = false; }
    if (ok && rt.dnnrtSync(handle)) { err = rt_error("dnnrtSync"); ok = false; }
    float total = 0.f;
    if (ok && rt.dnnrtEventElapsedMs(e0, e1, &total)) { err = rt_error("dnnrtEventElapsedMs"); ok = false; }
    for (size_t i = 0; ok && i < compute.size(); i++)
      if (c == class_of(compute[i])) ms[i] = total / (float)n;
  }
  rt.dnnrtEventDestroy(e0);
  rt.dnnrtEventDestroy(e1);
  return ok;
}

int64_t Session::algo_operand(const Op *op, int which, int64_t reference_value) const {
  const auto it = tuned.find(op);
  const int64_t id = it == tuned.end() ? 0 : (which ? it->second.second : it->second.first);
  if (id > 0) return DNNRT_CONV_ALGO_BASE + id;
  if (op->operands.back()->dtype != F32) return reference_value;
  const Value *filter = op->operands[which ? 5 : 1];
  bool direct = prog->direct_convolutions;
  for (size_t i = 0; !direct && !sparse_const.empty() && i < filter->uses.size(); i++) {  // the constant that is uploaded there
    const Op *copy = filter->uses[i].first;
    if (copy->kind != OP_MEMCPY || copy->mode != 1 || filter->uses[i].second != 0) continue;
    const Op *from = copy->operands[1]->def;
    direct = from && from->kind == OP_HOST_CONST && sparse_const.count(from->const_name);
  }
  return direct ? DNNRT_CONV_ALGO_DIRECT : reference_value;
}

// Convolutions with a call of their own; a block's launch has no variants.
bool Session::tunable(const Op *op) const {
  return (op->kind == OP_CONVFWD || op->kind == OP_CONV_BIAS_ACTIV || op->kind == OP_CONV_BIAS_ADD_ACTIV || op->kind == OP_CONV_ADD_CONV_ACTIV) &&
         !op->operands.empty() && op->operands.back()->dtype == F16 && !block_of.count(op);
}

std::vector<int64_t> Session::algos() const {
  std::vector<int64_t> out;
  for (const Op *op : prog->ops) {
    if (!launches(op)) continue;
    const auto it = tuned.find(op);
    out.push_back(it == tuned.end() ? 0 : it->second.first);
    out.push_back(it == tuned.end() ? 0 : it->second.second);
  }
  return out;
}

bool Session::set_algos(const int64_t *a, int64_t n, std::string &err) {
  std::vector<const Op *> compute;
  for (const Op *op : prog->ops)
    if (launches(op)) compute.push_back(op);
  if (!a || n != 2 * (int64_t)compute.size()) { err = "set_algos: two values per operation that launches are expected"; return false; }
  tuned.clear();
  for (size_t i = 0; i < compute.size(); i++) {
    if (a[2 * i] < 0 || a[2 * i + 1] < 0 || a[2 * i] >= 1000 || a[2 * i + 1] >= 1000) { err = "set_algos: a variant id is 0 .. 999"; return false; }
    if ((a[2 * i] || a[2 * i + 1]) && tunable(compute[i])) tuned[compute[i]] = {a[2 * i], a[2 * i + 1]};
  }
  drop_graphs();
  return true;
}

bool Session::tune(const void *const *inputs, int on_device, int reps, int64_t &changed, std::string &err) {
  changed = 0;
  if (mode != MODE_RESIDENT) { err = "tuning needs a resident session"; return false; }
  std::vector<const Op *> compute;
  for (const Op *op : prog->ops)
    if (launches(op)) compute.push_back(op);
  bool any = false;
  for (const Op *op : compute) any = any || tunable(op);
  if (host_backend || !prog->channels_last || !any) return true;
  std::vector<int32_t> ids((size_t)std::max(rt.dnnrtListConvTiles(nullptr, 0), 0));
  rt.dnnrtListConvTiles(ids.data(), (int32_t)ids.size());
  reps = std::max(reps, 3);
  const std::map<const Op *, std::pair<int64_t, int64_t>> before = tuned;
  // median per operation over `reps` profiled passes with the current choices
  auto measure = [&](std::vector<float> &med) -> bool {
    std::vector<std::vector<float>> runs;
    std::vector<float> ms;
    if (!profile_resident(inputs, on_device, false, ms, err)) return false;  // one pass to settle (code, caches)
    for (int r = 0; r < reps; r++) {
      if (!profile_resident(inputs, on_device, false, ms, err)) return false;
      runs.push_back(ms);
    }
    med.assign(compute.size(), 0.f);
    for (size_t i = 0; i < compute.size(); i++) {
      std::vector<float> v;
      for (const auto &r : runs) v.push_back(r[i]);
      std::sort(v.begin(), v.end());
      med[i] = v[v.size() / 2];
    }
    return true;
  };
  bool ok = true;
  for (int which = 0; which < 2 && ok; which++) {  // 0: every operation's (first) convolution; 1: the second one of the pairs
    std::vector<const Op *> targets;
    for (const Op *op : compute)
      if (tunable(op) && (which == 0 || op->kind == OP_CONV_ADD_CONV_ACTIV)) targets.push_back(op);
    if (targets.empty()) break;
    const auto chosen = tuned;  // what this round starts from
    auto with = [&](int64_t id) {
      tuned = chosen;
      for (const Op *op : targets) {
        auto &t = tuned[op];
        (which ? t.second : t.first) = id;
      }
    };
    std::vector<float> base;
    with(0);
    ok = measure(base);
    std::vector<float> best = base;
    std::vector<int64_t> best_id(compute.size(), 0);
    for (size_t c = 0; ok && c < ids.size(); c++) {
      std::vector<float> t;
      with(ids[c]);
      ok = measure(t);
      for (size_t i = 0; ok && i < compute.size(); i++)
        if (t[i] < best[i]) { best[i] = t[i]; best_id[i] = ids[c]; }
    }
    tuned = chosen;
    for (size_t i = 0; ok && i < compute.size(); i++) {
      if (std::find(targets.begin(), targets.end(), compute[i]) == targets.end()) continue;
      auto &t = tuned[compute[i]];
      (which ? t.second : t.first) = best[i] < 0.97f * base[i] ? best_id[i] : 0;
    }
  }
  if (!ok) { tuned = before; drop_graphs(); return false; }
  for (auto it = tuned.begin(); it != tuned.end();) {
    if (!it->second.first && !it->second.second) it = tuned.erase(it);
    else { changed++; ++it; }
  }
  drop_graphs();
  return true;
}

bool Session::set_conv_tile(int tile, std::string &err) {
  if (rt.dnnrtSetConvTile(handle, tile)) { err = rt_error("dnnrtSetConvTile"); return false; }
  drop_graphs();
  return true;
}

bool Session::sync(std::string &err) {
  if (rt.dnnrtSync(handle)) { err = rt_error("dnnrtSync"); return false; }
  return true;
}

}  // namespace dnnc
