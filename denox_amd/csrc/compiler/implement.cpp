#include "implement.hpp"
#include <algorithm>

namespace denox::compiler {

ComputeDispatch &ComputeDispatchBuilder::self() { return m_impl->m_edge.dispatches[m_index]; }

void ComputeDispatchBuilder::addBinding(dnx::Access access, TensorHandle t) {
  const auto &e = m_impl->m_edge;
  TensorBinding b;
  b.access = access;
  b.tensor = TensorId{static_cast<uint32_t>(t)};
  const bool isSrc = std::find(e.inputs.begin(), e.inputs.end(), t) != e.inputs.end();
  const bool isDst = e.output == t;
  if (isSrc && access == dnx::Access::ReadOnly) b.type = BindingType::Input;
  else if (isDst && access != dnx::Access::ReadOnly) b.type = BindingType::Output;
  else b.type = access == dnx::Access::ReadOnly ? BindingType::Read : BindingType::Write;
  self().bindings.push_back(b);
}

void ComputeDispatchBuilder::addBinding(dnx::Access access, TensorHandle t, Sym span) {
  addBinding(access, t);
  self().bindings.back().hasSpan = true;
  self().bindings.back().span = span;
}

void ComputeDispatchBuilder::addParamBinding(TensorId tensor) {
  TensorBinding b;
  b.access = dnx::Access::ReadOnly;
  b.tensor = tensor;
  b.type = BindingType::Param;
  self().bindings.push_back(b);
}

void ComputeDispatchBuilder::addPushConstant(Sym value, dnx::ScalarType dtype) { self().pushConstants.push_back(PushConstantDesc{value, dtype}); }

void ComputeDispatchBuilder::addTraversalFlag() {
  self().traversalFlagIndex = static_cast<int>(self().pushConstants.size());
  self().pushConstants.push_back(PushConstantDesc{Sym::Const(0), dnx::ScalarType::U32});
}

ComputeDispatchBuilder::~ComputeDispatchBuilder() {
  if (!m_impl) return;
  auto &bs = self().bindings;
  // kernels take their arguments in registration order within a class, classes in
  // the order Input < Output < Param < Read < Write
  std::stable_sort(bs.begin(), bs.end(), [](const TensorBinding &a, const TensorBinding &b) { return static_cast<int>(a.type) < static_cast<int>(b.type); });
  uint16_t n = 0;
  for (auto &b : bs) { b.set = 0; b.binding = n++; }
}

ComputeDispatchBuilder OpImpl::registerDispatch(hip::HipCompilerInstance kernel, const std::string &entryPoint, Sym wgX, Sym wgY, Sym wgZ,
                                                uint32_t bx, uint32_t by, uint32_t bz) {
  ComputeDispatch d;
  d.kernel = std::move(kernel);
  d.entryPoint = entryPoint;
  d.workgroupCountX = wgX; d.workgroupCountY = wgY; d.workgroupCountZ = wgZ;
  d.workgroupSize[0] = bx; d.workgroupSize[1] = by; d.workgroupSize[2] = bz;
  d.info.srcPath = d.kernel.sourcePath();
  m_edge.dispatches.push_back(std::move(d));
  return ComputeDispatchBuilder(m_edge.dispatches.size() - 1, this);
}

TensorId OpImpl::createParameter(size_t byteSize, dnx::ScalarType dtype, std::function<std::vector<uint8_t>()> value, uint16_t alignment) {
  SuperTensor t;
  t.byteSize = Sym::Const(static_cast<int64_t>(byteSize));
  t.alignment = alignment;
  t.isParam = true;
  t.type = dtype;
  t.format = dnx::TensorFormat::UNKNOWN;
  m_graph->tensors.push_back(std::move(t));
  TensorId id{static_cast<uint32_t>(m_graph->tensors.size() - 1)};
  m_edge.parameters.push_back(Parameter{id, std::move(value)});
  return id;
}

void OpImpl::createImplicitConcatConstrain(TensorHandle src0, TensorHandle src1, TensorHandle dst) {
  const size_t n = m_model->tensors().size();
  if (src0 < 0 || src1 < 0 || dst < 0 || static_cast<size_t>(src0) >= n || static_cast<size_t>(src1) >= n || static_cast<size_t>(dst) >= n)
    fail(Status::Internal, "Failed to create memory constrain, invalid node ids.");
  m_edge.memoryConstrains.push_back(MemoryConstrain{TensorId{static_cast<uint32_t>(src0)}, TensorId{static_cast<uint32_t>(src1)}, TensorId{static_cast<uint32_t>(dst)}});
}

void OpImpl::createViewConstrain(TensorHandle src, TensorHandle dst, uint64_t byteOffset) {
  const size_t n = m_model->tensors().size();
  if (src < 0 || dst < 0 || static_cast<size_t>(src) >= n || static_cast<size_t>(dst) >= n) fail(Status::Internal, "Failed to create memory constrain, invalid node ids.");
  m_edge.viewConstrains.push_back(ViewConstrain{TensorId{static_cast<uint32_t>(src)}, TensorId{static_cast<uint32_t>(dst)}, byteOffset});
}

ConcatView concatViewOf(const Model &model, TensorHandle t) {
  ConcatView v;
  const TensorNode &n = model.tensors()[static_cast<size_t>(t)];
  if (n.isInput || n.isOutput || n.consumers.size() != 1) return v;
  const Op &cat = model.ops()[static_cast<size_t>(n.consumers[0])];
  if (cat.kind != OpKind::Concat || cat.inputs.size() != 2 || cat.inputs[0] == cat.inputs[1]) return v;
  v.valid = true;
  v.concatOp = n.consumers[0];
  v.parent = cat.output;
  v.pitch = model.tensors()[static_cast<size_t>(cat.output)].channels;
  v.channelOffset = cat.inputs[0] == t ? 0 : model.tensors()[static_cast<size_t>(cat.inputs[0])].channels;
  return v;
}

void OpImpl::finish() { m_graph->edges.push_back(std::move(m_edge)); }

dnx::TensorFormat interfaceFormat(const std::vector<InterfaceTensorDescriptor> &descs, const std::string &name, size_t index) {
  for (const auto &d : descs) if (d.name == name) return d.format;
  if (index < descs.size() && descs[index].name.empty()) return descs[index].format;
  return dnx::TensorFormat::SSBO_HWC;
}

void markBlockedInterface(Model &model, const CompileOptions &opt) {
  if (!opt.features.enableBlockedLayout) return;
  auto mark = [&](const std::vector<TensorHandle> &list, const std::vector<InterfaceTensorDescriptor> &descs) {
    for (size_t i = 0; i < list.size(); ++i) {
      const TensorNode &n = model.tensors()[static_cast<size_t>(list[i])];
      if (interfaceFormat(descs, n.name, i) != dnx::TensorFormat::SSBO_CHWC8 || n.channels % 8 || (n.isInput && n.isOutput)) continue;
      if (n.isOutput && !n.consumers.empty()) continue;
      if (std::count(list.begin(), list.end(), list[i]) != 1) continue;
      model.setBlockedInterface(list[i]);
    }
  };
  mark(model.inputs(), opt.inputDescriptors);
  mark(model.outputs(), opt.outputDescriptors);
}

ComputeDispatch relayoutDispatch(const hip::HipCompiler &hipc, SymGraph &sym, const TensorNode &n, Sym bytes, dnx::TensorFormat from, dnx::TensorFormat to, uint32_t src, uint32_t dst) {
  auto layoutId = [](dnx::TensorFormat f) -> int {
    switch (f) {
    case dnx::TensorFormat::SSBO_HWC: return 0;
    case dnx::TensorFormat::SSBO_CHW: return 1;
    case dnx::TensorFormat::SSBO_CHWC8: return 2;
    default: fail(Status::Unsupported, "interface tensors must be SSBO_HWC, SSBO_CHW or SSBO_CHWC8");
    }
  };
  if ((from == dnx::TensorFormat::SSBO_CHWC8 || to == dnx::TensorFormat::SSBO_CHWC8) && n.channels % 8) fail(Status::InvalidArgument, "CHWC8 needs a channel count divisible by 8");
  ComputeDispatch d;
  d.kernel = hipc.read("relayout.hip");
  d.kernel.define("CH", n.channels); d.kernel.define("SRC_LAYOUT", layoutId(from)); d.kernel.define("DST_LAYOUT", layoutId(to));
  d.entryPoint = "relayout_c" + std::to_string(n.channels) + "_" + std::to_string(layoutId(from)) + "to" + std::to_string(layoutId(to));
  d.kernel.define("KERNEL_NAME", d.entryPoint);
  // HWC <-> CHWC8 moves one 16-byte vector per thread, HWC <-> CHW of whole 8-channel groups a tile of pixels per workgroup (MODE_BLOCK),
  // every other pair one pixel per thread (see relayout.hip)
  const bool blocky = from != dnx::TensorFormat::SSBO_CHW && to != dnx::TensorFormat::SSBO_CHW && n.channels % 8 == 0;
  const bool hwc = from == dnx::TensorFormat::SSBO_HWC || to == dnx::TensorFormat::SSBO_HWC, chw = from == dnx::TensorFormat::SSBO_CHW || to == dnx::TensorFormat::SSBO_CHW;
  const int64_t tile = hwc && chw && n.channels % 8 == 0 && n.channels <= 256 ? (n.channels <= 32 ? 512 : n.channels <= 64 ? 256 : n.channels <= 128 ? 128 : 64) : 256;
  d.workgroupCountX = sym.cdiv(sym.mul(sym.mul(n.width, n.height), blocky ? static_cast<int64_t>(n.channels / 8) : 1), tile);
  d.workgroupCountY = d.workgroupCountZ = Sym::Const(1);
  d.workgroupSize[0] = 256;
  d.bindings = {TensorBinding{0, 0, dnx::Access::ReadOnly, TensorId{src}, BindingType::Input, false, Sym::Const(0)},
                TensorBinding{0, 1, dnx::Access::WriteOnly, TensorId{dst}, BindingType::Output, false, Sym::Const(0)}};
  d.pushConstants = {PushConstantDesc{n.width, dnx::ScalarType::U32}, PushConstantDesc{n.height, dnx::ScalarType::U32}};
  d.info.name = "relayout"; d.info.operation = "relayout"; d.info.srcPath = "relayout.hip";
  d.info.hasReads = d.info.hasWrites = d.info.hasFlops = true;
  d.info.memoryReads = d.info.memoryWrites = bytes;
  d.info.flops = Sym::Const(0);
  return d;
}

SuperGraph implement(const Model &model, SymGraph &sym, const std::vector<std::unique_ptr<IShader>> &shaders, const hip::HipCompiler &hipc, const CompileOptions &opt) {
  SuperGraph g;
  g.tensors.reserve(model.tensors().size() + 64);
  for (size_t i = 0; i < model.tensors().size(); ++i) {
    const TensorNode &t = model.tensors()[i];
    SuperTensor st;
    st.byteSize = sym.mul(sym.mul(t.width, t.height), static_cast<int64_t>(t.channels) * 2);
    st.alignment = 256;
    st.modelTensor = static_cast<int>(i);
    st.name = t.name;
    g.tensors.push_back(std::move(st));
  }
  // the same tensors stored channel-block-major
  const size_t N = model.tensors().size();
  g.modelTensorCount = N;
  for (size_t i = 0; i < N; ++i) {
    SuperTensor st = g.tensors[i];
    st.format = dnx::TensorFormat::SSBO_CHWC8;
    g.tensors.push_back(std::move(st));
  }
  for (const auto &shader : shaders) {
    for (const Match &m : shader->matchAll(model, opt)) {
      for (unsigned config : shader->acceptMatch(model, m, opt)) {
        OpImpl impl(&g, &model, m.inputs, m.output, m.ops);
        impl.edge().shader = shader->name();
        impl.edge().speedup = shader->speedup(config);
        impl.edge().outputVariant = m.outputVariant;
        impl.edge().inputVariants = m.inputVariants;
        impl.edge().outputFormat = m.outputFormat;
        impl.edge().inputFormats = m.inputFormats;
        shader->implement(impl, model, m, config, sym, opt);
        if (m.blocked()) {
          // The shaders bind model tensors by handle; an input or output the match takes in CHWC8 is that tensor's second
          // super-graph tensor.
          auto blockedTensor = [&](uint32_t t) -> uint32_t {
            if (t >= N) return t; // a parameter
            if (static_cast<int>(t) == m.output && m.outputFormat) return t + static_cast<uint32_t>(N);
            for (size_t i = 0; i < m.inputs.size(); ++i)
              if (m.inputs[i] == static_cast<int>(t) && i < m.inputFormats.size() && m.inputFormats[i]) return t + static_cast<uint32_t>(N);
            return t;
          };
          for (auto &d : impl.edge().dispatches)
            for (auto &b : d.bindings) b.tensor.index = blockedTensor(b.tensor.index);
          for (auto &mc : impl.edge().memoryConstrains) {
            mc.src0.index = blockedTensor(mc.src0.index);
            mc.src1.index = blockedTensor(mc.src1.index);
            mc.dst.index = blockedTensor(mc.dst.index);
          }
        }
        impl.finish();
      }
    }
  }
  // an interface tensor kept in CHWC8 may also be converted
  for (size_t i = 0; i < N; ++i) {
    const TensorNode &n = model.tensors()[i];
    if (!n.blockedInterface) continue;
    const uint32_t hwc = static_cast<uint32_t>(i), blocked = static_cast<uint32_t>(i + N);
    SuperGraphEdge e;
    e.inputs = {static_cast<int>(i)};
    e.output = static_cast<int>(i);
    e.shader = "relayout";
    e.config = n.isInput ? "chwc8>hwc" : "hwc>chwc8";
    e.inputFormats = {n.isInput ? 1 : 0};
    e.outputFormat = n.isInput ? 0 : 1;
    e.dispatches.push_back(n.isInput ? relayoutDispatch(hipc, sym, n, g.tensors[i].byteSize, dnx::TensorFormat::SSBO_CHWC8, dnx::TensorFormat::SSBO_HWC, blocked, hwc)
                                     : relayoutDispatch(hipc, sym, n, g.tensors[i].byteSize, dnx::TensorFormat::SSBO_HWC, dnx::TensorFormat::SSBO_CHWC8, hwc, blocked));
    g.edges.push_back(std::move(e));
  }
  return g;
}

} // namespace denox::compiler
