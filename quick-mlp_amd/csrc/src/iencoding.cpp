#include <qmlp/iencoding.h>

#include <qmlp/encoding_hashgrid.h>
#include <qmlp/encoding_line_integration.h>
#include <qmlp/encoding_identity.h>
#include <qmlp/qmlp.h>
#include <qmlp_hip.h>

#include <cctype>
#include <cstring>
#include <mutex>

QUICKMLP_NAMESPACE_BEGIN

namespace {

// Kernel arguments of the standalone kernels: fixed ones plus the optional parameter struct.
struct ArgPack
{
    std::vector<void*> ptrs;
    std::vector<char> paramBytes;
};

std::string standaloneSource(const IEncoding& e, const std::string& callForward, const std::string& callAdjoint,
                             const std::string& callCorners = "", const std::string& callScatter = "",
                             const std::string& callTraceGather = "", const std::string& callTraceScatter = "", int groups = 1, bool sharedTile = false, bool byLevels = false)
{
    auto kl = QuickMLP::Instance().kernelLoader();
    std::string codeTemplate = kl->findFile("qmlp/kernels/encoding_kernels.h").value();
    std::stringstream includes;
    e.fillCode(includes);
    includes << "\n";
    replaceAll(codeTemplate, "$$INCLUDES$$", includes.str());
    replaceAll(codeTemplate, "$$ENCODING_PARAMETERS$$",
               e.hasParameters() ? ", const " + e.parameterName() + " cEncoding" : std::string());
    replaceAll(codeTemplate, "$$SHARED_TILE$$", sharedTile ? "1" : "0");
    replaceAll(codeTemplate, "$$BY_LEVELS$$", byLevels ? "1" : "0");
    if (byLevels) {
        std::string tiles;
        for (int perWave : e.levelTiles()) tiles += (tiles.empty() ? "" : ", ") + std::to_string(perWave);
        replaceAll(codeTemplate, "$$ENCODING$$", e.qualifiedName());
        replaceAll(codeTemplate, "$$LEVEL_TILES$$", tiles);
    }
    // the channels of a group of levels (EncodingForwardKernel)
    const std::string levels = std::to_string(e.numOutputChannels() / e.channelsWrittenTogether());
    const std::string features = std::to_string(e.channelsWrittenTogether());
    replaceAll(codeTemplate, "$$LEVEL_GROUPS$$", std::to_string(groups));
    replaceAll(codeTemplate, "$$GROUP_CHANNELS$$", groups == 1 ? std::to_string(e.numOutputChannels())
                                                               : "(" + levels + " + GROUPS - 1) / GROUPS * " + features);
    replaceAll(codeTemplate, "$$FIRST_CHANNEL$$", groups == 1 ? "0" : levels + " * group / GROUPS * " + features);
    replaceAll(codeTemplate, "$$CHANNELS$$", groups == 1 ? "CHANNELS" : levels + " * (group + 1) / GROUPS * " + features + " - firstChannel");
    replaceAll(codeTemplate, "$$CALL_ENCODINGS_FORWARD$$", callForward);
    replaceAll(codeTemplate, "$$CALL_ENCODINGS_ADJOINT$$", callAdjoint);
    replaceAll(codeTemplate, "$$CALL_ENCODINGS_CORNERS$$", callCorners);
    replaceAll(codeTemplate, "$$CALL_ENCODINGS_SCATTER$$", callScatter);
    replaceAll(codeTemplate, "$$CALL_ENCODINGS_TRACE_GATHER$$", callTraceGather);
    replaceAll(codeTemplate, "$$CALL_ENCODINGS_TRACE_SCATTER$$", callTraceScatter);
    return codeTemplate;
}

} // namespace

std::string IEncoding::forwardKernelSource(int groups) const
{
    std::stringstream call;
    if (groups > 1) call << qualifiedName() << "::forwardGroup<0, GROUPS>(group, encodingInput, encodingOutput";
    else call << qualifiedName() << "::forward(encodingInput, encodingOutput";
    if (hasParameters()) call << ", cEncoding";
    call << ");\n";
    return standaloneSource(*this, call.str(), "", "", "", "", "", groups);
}

std::vector<KernelFunction> IEncoding::compileForwardByLevels(int flags) const
{
    return QuickMLP::Instance().kernelLoader()->getKernels({"qmlp::kernel::EncodingLevelsKernel", "qmlp::kernel::EncodingRowsKernel"},
                                                           standaloneSource(*this, "", "", "", "", "", "", 1, false, true), flags);
}

std::string IEncoding::adjointKernelSource(int adjointMode, bool sharedTile) const
{
    const bool hasInputGradients = adjointMode & INPUT_GRADIENTS;
    const bool hasParamGradients = (adjointMode & PARAM_GRADIENTS) && hasParameters();
    if (sharedTile) {
        std::string source = standaloneSource(*this, "", "", "", "", "", "", 1, true);
        replaceAll(source, "$$ENCODING$$", qualifiedName());
        replaceAll(source, "$$SHARED_WAVES$$", std::to_string(sharedAdjointWaves()));
        replaceAll(source, "$$INPUT_GRADIENTS$$", hasInputGradients ? "true" : "false");
        replaceAll(source, "$$PARAMETER_GRADIENTS$$", hasParamGradients ? "true" : "false");
        return source;
    }
    // encodings with a tile-wide scatter take their parameter gradients out of the per-point call
    std::stringstream call, scatter;
    call << qualifiedName() << "::template adjoint<" << (hasInputGradients ? "true" : "false") << ", "
         << (hasParamGradients ? "!" + qualifiedName() + "::HasTileScatter" : std::string("false"))
         << ">(encodingInput, encodingAdjOutput, encodingAdjInput";
    if (hasParameters()) call << ", cEncoding";
    call << ");\n";
    if (hasParamGradients)
        scatter << "if constexpr (" << qualifiedName() << "::HasTileScatter)\n            " << qualifiedName()
                << "::scatterTile(lane, tileBase, numel, inputs, [&](int pt, int c) { return adjOutputs.data_[(tileBase + pt)"
                   " * adjOutputs.strides_[0] + static_cast<long long>(c) * adjOutputs.strides_[1]]; }, cEncoding);\n";
    return standaloneSource(*this, "", call.str(), "", scatter.str());
}

void IEncoding::precompile(int adjointMode)
{
    auto kl = QuickMLP::Instance().kernelLoader();
    const int flags = QuickMLP::Instance().getCompileFlags() | KernelLoader::CompileOnly;
    kl->getKernel("qmlp::kernel::EncodingForwardKernel", forwardKernelSource(1), flags);
    if (levelGroups() > 1) kl->getKernel("qmlp::kernel::EncodingForwardKernel", forwardKernelSource(levelGroups()), flags);
    if (!levelTiles().empty() && numOutputChannels() <= kernel::ENCODING_ROWS_MAX_CHANNELS) compileForwardByLevels(flags);
    if (adjointMode > 0) {
        CHECK_ERROR(adjointMode <= ALL_GRADIENTS, "Illegal adjoint mode");
        kl->getKernel("qmlp::kernel::EncodingAdjointKernel", adjointKernelSource(adjointMode), flags);
        if (sharedAdjointWaves() > 0) kl->getKernel("qmlp::kernel::EncodingAdjointSharedKernel", adjointKernelSource(adjointMode, true), flags);
        if (const auto* layout = (adjointMode & PARAM_GRADIENTS) && hasParameters() ? sliceLayout(true) : nullptr) {
            for (int v = 0; v < recordsVariants(*layout); ++v) compileRecords(*layout, adjointMode & INPUT_GRADIENTS, v, flags);
            compileSlices(*layout, flags);
        }
    }
}

bool IEncoding::forwardByLevels(const Tensor& input, const Tensor& output) const
{
    const long long numel = input.size(0);
    const std::vector<int> levels = levelTiles();
    if (levels.empty() || numOutputChannels() > kernel::ENCODING_ROWS_MAX_CHANNELS) return false;
    // Tables that one die's L2 (4 MB) would have to take turns with, and batches that make up for a second kernel. The time of the kernel of whole
    // rows grows in steps of a workgroup of 256 points per compute unit (2^16 points of 256), and just before the end of the first two its
    // wavefronts walk through the levels together. Whole rows -> by levels, us:
    //   2^14 / 2^15 points   13 -> 17 / 23 -> 24 (16 levels of 2^19 entries of 2 floats, 50 MB; of 2 halves 10 -> 14 / 17 -> 20)
    //   3 2^14, 2^16         37 -> 30, 42 -> 37 (halves 33 -> 25, 35 -> 29), but with 128 bytes or more per point and level 62 -> 68 (16 levels of
    //                        8 halves, 2^16), 53 -> 58 (12 of 8 floats), 42 -> 48 (4-D, 12 of 2 floats)
    //   9 2^13, 7 2^14       66 -> 40, 72 -> 57 (halves 53 -> 32, 52 -> 43; 16 of 8 halves 105 -> 84, 117 -> 111)
    //   15 2^13, 2^17        72 -> 60, 70 -> 63, in a training step 67 -> 67 (halves 50 -> 46, 49 -> 49, 12 levels 45 -> 44, 45 -> 47; 4-D 86 -> 83, 81 -> 88)
    //   2^18 / 2^20          183 -> 116 / 776 -> 434 (halves 133 -> 95 / 569 -> 361; 16 of 8 halves 265 -> 236 / 1139 -> 949)
    // One feature per level: 66 -> 48 at 3 2^15 points, but 78 -> 86 at 3 2^16. Tables of 13 MB at 2^17 points: 44 -> 56. Eight levels, one per die, of
    // which the coarse ones are done first: 2^16 / 2^17 / 2^18 points 25 -> 29 / 39 -> 50 / 78 -> 90 (of 2 floats), 45 -> 59 / 92 -> 109 / 189 -> 211 (8
    // floats), 26 -> 32 / 41 -> 54 / 97 -> 97 (4 halves); ten 27 -> 22 / 38 -> 38 / 71 -> 70 (2 halves).
    constexpr long long MIN_TABLE_BYTES = 20 << 20, POINTS_PER_WORKGROUP = 256;
    constexpr int MIN_LEVELS = 10, WIDE_BYTES = 128;
    const long long tableBytes = static_cast<long long>(parameterCount()) * (parameterPrecision(Tensor::INFERENCE) == Tensor::HALF ? 2 : 4);
    if (static_cast<int>(levels.size()) < MIN_LEVELS || numel < FORWARD_WHOLE_ROWS_MIN_BATCH || tableBytes < MIN_TABLE_BYTES) return false;
    const long long step = POINTS_PER_WORKGROUP * KernelFunction::computeUnits();
    if (numel <= step && 4 * gatherRegistersPerPoint() >= WIDE_BYTES) return false;
    if (4 * numel > 7 * step && numel <= 2 * step) return false;
    if (channelsWrittenTogether() < 2 && numel < 4 * step) return false;
    if (numel * numOutputChannels() >= (1ll << 32)) return false;   // (lanes of a launch)
    // Rows without gaps, which hold other points' values between the two kernels: not those that a caller reads the positions from.
    if (output.size(1) != numOutputChannels() || output.strides()[0] != numOutputChannels()) return false;
    const float* rows = static_cast<const float*>(output.rawPtr());
    const float *first = static_cast<const float*>(input.rawPtr()), *last = first;
    for (int d = 0; d < 2; ++d) {
        const long long extent = (input.size(d) - 1ll) * input.strides()[d];
        (extent < 0 ? first : last) += extent;
    }
    return last < rows || rows + numel * numOutputChannels() <= first;
}

std::string IEncoding::forwardKernelName(const Tensor& input, const Tensor& output) const
{
    return forwardByLevels(input, output) ? "EncodingLevelsKernel" : "EncodingForwardKernel";
}

void IEncoding::forward(const Tensor& input, Tensor& output, stream_t stream,
                        const std::optional<const Tensor>& parametersForward)
{
    CHECK_DIM(input, 2);
    CHECK_DIM(output, 2);
    CHECK_DTYPE(input, Tensor::FLOAT);
    CHECK_DTYPE(output, Tensor::FLOAT);
    CHECK_SIZE(output, 0, input.size(0));
    CHECK_ERROR(input.size(1) > maxInputChannel());
    CHECK_ERROR(output.size(1) >= numOutputChannels());
    CHECK_ERROR(output.strides()[1] == 1, "The output stride along the channels must be 1");
    long long numel = input.size(0);
    if (hasParameters())
        CHECK_ERROR((parametersForward.has_value() && parametersForward.value().defined()) || hasParameterTensor(Tensor::INFERENCE),
                    "The encoding has parameters, but no inference tensor is bound or passed");
    if (numel == 0) return;

    const bool byLevels = forwardByLevels(input, output);
    const int groups = numel < FORWARD_WHOLE_ROWS_MIN_BATCH ? levelGroups() : 1;
    auto& kernel = forwardKernel_[groups > 1 ? 1 : 0];
    if (byLevels) {
        static std::mutex mutex;
        std::lock_guard<std::mutex> lock(mutex);
        if (forwardByLevels_.empty()) forwardByLevels_ = compileForwardByLevels(QuickMLP::Instance().getCompileFlags());
    } else if (!kernel.has_value()) {
        kernel = QuickMLP::Instance().kernelLoader()->getKernel(
            "qmlp::kernel::EncodingForwardKernel", forwardKernelSource(groups), QuickMLP::Instance().getCompileFlags()).value();
    }

    std::vector<char> paramBytes(4096);
    if (hasParameters()) {
        if (parametersForward.has_value()) setParameter(parametersForward.value(), Tensor::INFERENCE);
        int n = fillParameterMemory(paramBytes.data(), static_cast<int>(paramBytes.size()));
        (void)n;
    }

    const int block = 256;
    auto inputAcc = input.accessor<kernel::Tensor2Read<float>>();
    auto outputAcc = output.accessor<kernel::Tensor2RW<float>>();
    if (byLevels) {
        const long long tiles = divUp<long long>(numel, 64);
        long long workgroups = 0;
        for (int perWave : levelTiles()) workgroups += divUp<long long>(tiles, perWave * kernel::ENCODING_LEVEL_WAVES);
        const long long perDie = divUp<long long>(workgroups, kernel::DIES);
        float* rows = outputAcc.data_;
        std::vector<void*> levelArgs = {&numel, &inputAcc, &rows, paramBytes.data()}, rowArgs = {&numel, &rows};
        forwardByLevels_[0].launch(static_cast<int>(kernel::DIES * perDie), block, 0, stream, levelArgs.data());
        forwardByLevels_[1].launch(static_cast<int>(tiles), 64, 0, stream, rowArgs.data());
    } else {
        auto& fun = kernel.value();
        const int grid = groups * static_cast<int>(std::min<long long>(divUp<long long>(numel, block), std::max(1, fun.fullGridSize(block, 0) / groups)));
        std::vector<void*> args = {&numel, &inputAcc, &outputAcc};
        if (hasParameters()) args.push_back(paramBytes.data());
        fun.launch(grid, block, 0, stream, args.data());
    }

    if (hasParameters() && parametersForward.has_value()) setParameter({}, Tensor::INFERENCE);
}

void IEncoding::adjoint(const Tensor& input, const Tensor& adjOutput, Tensor& adjInput, stream_t stream,
                        const std::optional<const Tensor>& parametersForward,
                        const std::optional<const Tensor>& parametersGradients, int adjointMode)
{
    adjoint(input, adjOutput, adjInput, stream, parametersForward, parametersGradients, adjointMode, nullptr);
}

void IEncoding::adjoint(const Tensor& input, const Tensor& adjOutput, Tensor& adjInput, stream_t stream,
                        const std::optional<const Tensor>& parametersForward,
                        const std::optional<const Tensor>& parametersGradients, int adjointMode, void* tmpMemory, bool overwriteParameters)
{
    CHECK_DIM(input, 2);
    CHECK_DIM(adjOutput, 2);
    CHECK_DIM(adjInput, 2);
    CHECK_DTYPE(input, Tensor::FLOAT);
    CHECK_DTYPE(adjOutput, Tensor::FLOAT);
    CHECK_DTYPE(adjInput, Tensor::FLOAT);
    CHECK_SIZE(adjOutput, 0, input.size(0));
    CHECK_SIZE(adjInput, 0, input.size(0));
    CHECK_ERROR(input.size(1) > maxInputChannel());
    CHECK_ERROR(adjOutput.size(1) >= numOutputChannels());
    CHECK_ERROR(adjInput.size(1) == input.size(1));
    CHECK_ERROR(adjointMode >= 1 && adjointMode <= ALL_GRADIENTS, "Illegal adjoint mode");
    long long numel = input.size(0);
    if (hasParameters()) {
        CHECK_ERROR((parametersForward.has_value() && parametersForward.value().defined()) || hasParameterTensor(Tensor::INFERENCE),
                    "The encoding has parameters, but no inference tensor is bound or passed");
        CHECK_ERROR(!(adjointMode & PARAM_GRADIENTS) || (parametersGradients.has_value() && parametersGradients.value().defined())
                        || hasParameterTensor(Tensor::GRADIENTS),
                    "Parameter gradients requested, but no gradient tensor is bound or passed");
    }
    const bool bySlices = tmpMemory != nullptr && adjointMemory(numel, adjointMode) > 0;
    CHECK_ERROR(bySlices || !overwriteParameters, "adjoint() adds to parameter gradients of this batch that it was asked to overwrite");
    if (numel == 0) return;

    const bool sharedTile = !bySlices && sharedAdjointWaves() > 0 && numel <= SHARED_ADJOINT_MAX_BATCH;
    auto& kernel = sharedTile ? adjointSharedKernel_[adjointMode] : adjointKernel_[adjointMode];
    if (!bySlices && !kernel.has_value())
        kernel = QuickMLP::Instance().kernelLoader()->getKernel(
            sharedTile ? "qmlp::kernel::EncodingAdjointSharedKernel" : "qmlp::kernel::EncodingAdjointKernel",
            adjointKernelSource(adjointMode, sharedTile), QuickMLP::Instance().getCompileFlags()).value();

    std::vector<char> paramBytes(4096);
    if (hasParameters()) {
        if (parametersForward.has_value()) setParameter(parametersForward.value(), Tensor::INFERENCE);
        if (parametersGradients.has_value()) setParameter(parametersGradients.value(), Tensor::GRADIENTS);
        int n = fillParameterMemory(paramBytes.data(), static_cast<int>(paramBytes.size()));
        (void)n;
    }

    if (bySlices) {
        adjointBySlices(*sliceLayout(true), input, adjOutput, adjInput, stream, adjointMode, tmpMemory, paramBytes.data(), overwriteParameters);
    } else {
        auto& fun = kernel.value();
        const int block = sharedTile ? sharedAdjointWaves() * 64 : 256;
        const int grid = static_cast<int>(std::min<long long>(divUp<long long>(numel, sharedTile ? 64 : block), fun.fullGridSize(block, 0)));
        auto inputAcc = input.accessor<kernel::Tensor2Read<float>>();
        auto adjOutputAcc = adjOutput.accessor<kernel::Tensor2Read<float>>();
        auto adjInputAcc = adjInput.accessor<kernel::Tensor2RW<float>>();
        std::vector<void*> args = {&numel, &inputAcc, &adjOutputAcc, &adjInputAcc};
        if (hasParameters()) args.push_back(paramBytes.data());
        fun.launch(grid, block, 0, stream, args.data());
    }

    if (hasParameters() && parametersForward.has_value()) setParameter({}, Tensor::INFERENCE);
    if (hasParameters() && parametersGradients.has_value()) setParameter({}, Tensor::GRADIENTS);
}

size_t IEncoding::adjointMemory(long long numel, int adjointMode) const
{
    if (!(adjointMode & PARAM_GRADIENTS) || !hasParameters() || numel >= (1 << 27)) return 0;
    const auto* layout = sliceLayout(true);
    return layout && slicesPay(*layout, numel, adjointMode & INPUT_GRADIENTS ? SLICE_GRADIENTS_MIN_BATCH_STANDALONE_INPUT
                                                                               : SLICE_GRADIENTS_MIN_BATCH_STANDALONE) ? layout->workspaceBytes(numel) : 0;
}

int IEncoding::recordsVariants(const GradientSliceLayout& layout)
{
    int n = 1;
    while ((layout.pointsPerWorkgroup >> n) >= 128) ++n;
    return n;
}

std::optional<KernelFunction> IEncoding::compileRecords(const GradientSliceLayout& layout, bool inputGradients, int variant, int flags) const
{
    std::stringstream source;
    fillCode(source);
    source << "\n" << KernelLoader::MainFile("qmlp/kernels/grid_gradient.h");
    return QuickMLP::Instance().kernelLoader()->getKernel(
        format("qmlp::kernel::GridGradientRecordsKernel<%s, 0, 0, %d, %d, %d, %d>", layout.configType.c_str(), layout.sliceFloats,
               layout.pointsPerWorkgroup >> variant, inputGradients ? 1 : 0, layout.levelGroups(inputGradients ? GradientSliceLayout::FROM_ENTRIES : GradientSliceLayout::NO_INPUT_GRADIENTS)),
        source.str(), flags);
}

std::vector<KernelFunction> IEncoding::compileSlices(const GradientSliceLayout& layout, int flags) const
{
    std::stringstream source;
    fillCode(source);
    source << "\n" << KernelLoader::MainFile("qmlp/kernels/grid_gradient.h");
    return QuickMLP::Instance().kernelLoader()->getKernels(
        {format("qmlp::kernel::GridGradientSlicesKernel<%s, %d, true>", layout.configType.c_str(), layout.sliceFloats),
         format("qmlp::kernel::GridGradientExceptionsKernel<%s, 0, 0, %d>", layout.configType.c_str(), layout.sliceFloats)},
        source.str(), flags);
}

void IEncoding::adjointBySlices(const GradientSliceLayout& layout, const Tensor& input, const Tensor& adjOutput, Tensor& adjInput, stream_t stream,
                                int adjointMode, void* tmpMemory, char* parameters, bool overwriteParameters)
{
    CHECK_ERROR(reinterpret_cast<uintptr_t>(tmpMemory) % 256 == 0, "The temporary memory must be aligned to 256 bytes");
    auto& sk = sliceKernels_;
    const int flags = QuickMLP::Instance().getCompileFlags();
    int numel = static_cast<int>(input.size(0));
    const bool inputGradients = adjointMode & INPUT_GRADIENTS;
    const auto inputFrom = inputGradients ? GradientSliceLayout::FROM_ENTRIES : GradientSliceLayout::NO_INPUT_GRADIENTS;
    const int groups = layout.levelGroups(inputFrom);
    // as for the fused networks: as many points per workgroup as keep every compute unit busy
    int variant = 0;
    while (variant + 1 < recordsVariants(layout) && groups * divUp(numel, layout.pointsPerWorkgroup >> variant) < KernelFunction::computeUnits()) ++variant;
    auto& variants = sk.records[inputGradients ? 1 : 0];
    if (variants.empty()) variants.resize(recordsVariants(layout));
    if (!variants[variant].has_value()) variants[variant] = compileRecords(layout, inputGradients, variant, flags).value();
    if (!sk.slices.has_value()) {
        const auto kernels = compileSlices(layout, flags);
        sk.items = Tensor(Tensor::FLOAT, {static_cast<int32_t>(layout.items.size() * (sizeof(GradientSlice) / sizeof(float)))});
        QMLP_HIP_CALL(qmlp_hip_memcpy_h2d(sk.items.rawPtr(), layout.items.data(), layout.items.size() * sizeof(layout.items[0]), nullptr));
        sk.exceptions = kernels.at(1);
        sk.slices = kernels.at(0);   // (last: what it reads is there, whatever of the above has thrown)
    }

    const int points = layout.pointsPerWorkgroup >> variant;
    GradientWorkspace workspace = layout.workspace(tmpMemory, numel, points, inputFrom);
    int overwrite = overwriteParameters ? 1 : 0, overwriteInput = 0;
    auto inputAcc = input.accessor<kernel::Tensor2Read<float>>();
    auto adjOutputAcc = adjOutput.accessor<kernel::Tensor2Read<float>>();
    {
        auto adjInputAcc = adjInput.accessor<kernel::Tensor2RW<float>>();
        const void* derivatives = nullptr;
        void* args[] = {&numel, &inputAcc, &adjOutputAcc, parameters, &workspace, &overwrite, &adjInputAcc, &overwriteInput, &derivatives};
        variants[variant].value().launch(layout.workgroupsPerRegion(inputFrom) * layout.regionSlots(numel, points), points,
                                         layout.recordsLdsBytes(points), stream, args);
    }
    {
        float* gradients = nullptr;
        std::memcpy(&gradients, parameters + sizeof(void*), sizeof(void*));   // HashGridParams: forward table, gradient table, ...
        const void* items = sk.items.rawPtr();
        void* args[] = {&numel, &workspace, &gradients, &items, &overwrite};
        sk.slices.value().launch(static_cast<int>(layout.items.size()), 1024, layout.slicesLdsBytes(), stream, args);
    }
    void* args[] = {&inputAcc, &adjOutputAcc, parameters, &workspace};
    sk.exceptions.value().launch(layout.exceptionsGrid(workspace), layout.EXCEPTIONS_BLOCK, 0, stream, args);
}

void EncodingHashGrid::corners(const Tensor& input, unsigned* indices, float* weights, stream_t stream, int mode)
{
    CHECK_DIM(input, 2);
    CHECK_DTYPE(input, Tensor::FLOAT);
    CHECK_ERROR(input.size(1) > maxInputChannel());
    CHECK_ERROR(mode >= 0 && mode <= 4, "mode 0: the index function, 1: the gathers of the forward pass, 2: the gradient scatter, "
                                        "3: the gradient records of the slice kernels, 4: the sums of the column kernel");
    CHECK_ERROR(mode != 2 || (numFeaturesPerLevel_ & (numFeaturesPerLevel_ - 1)) == 0 && numFeaturesPerLevel_ <= 32,
                "the tile-wide gradient scatter exists for 1, 2, 4 .. 32 features per level");
    CHECK_ERROR(mode == 0 || hasParameterTensor(Tensor::INFERENCE), "the traces read the table: bind one first");
    long long numel = input.size(0);
    if (numel == 0) return;
    if (!cornersKernel_[mode].has_value()) precompileCorners(mode, false);
    auto& fun = cornersKernel_[mode].value();
    std::vector<char> paramBytes(4096);
    int n = fillParameterMemory(paramBytes.data(), static_cast<int>(paramBytes.size()));
    (void)n;
    const int block = 256;
    // modes 0 and 1: a lane per point; mode 2: a wavefront per 64 points
    const int grid = static_cast<int>(std::min<long long>(divUp<long long>(numel, block), fun.fullGridSize(block, 0)));
    auto inputAcc = input.accessor<kernel::Tensor2Read<float>>();
    int perPoint = numLevels() * (1 << ndim());
    if (mode == 3 || mode == 4) {
        void* args[] = {&numel, &inputAcc, &indices, &weights, paramBytes.data()};
        fun.launch(grid, block, 0, stream, args);
        return;
    }
    void* args[] = {&numel, &inputAcc, &indices, &weights, &perPoint, paramBytes.data()};
    fun.launch(grid, block, 0, stream, args);
}

void EncodingHashGrid::precompileCorners(int mode, bool compileOnly)
{
    CHECK_ERROR(mode >= 0 && mode <= 4, "mode 0: the index function, 1: the gathers of the forward pass, 2: the gradient scatter, "
                                        "3: the gradient records of the slice kernels, 4: the sums of the column kernel");
    if (mode == 3) {
        // the record building of kernels/grid_gradient.h with the slice size the fused network uses for this grid
        GradientSliceLayout layout;
        CHECK_ERROR(gradientSlices(layout, false), "this grid has no gradient slices");
        std::stringstream source;
        fillCode(source);
        source << "\n" << KernelLoader::MainFile("qmlp/kernels/grid_gradient.h");
        const int flags = QuickMLP::Instance().getCompileFlags() | (compileOnly ? KernelLoader::CompileOnly : 0);
        auto kernel = QuickMLP::Instance().kernelLoader()->getKernel(
            "qmlp::kernel::GridGradientTraceKernel<" + layout.configType + ", " + std::to_string(layout.sliceFloats) + ">",
            source.str(), flags);
        if (!compileOnly) cornersKernel_[mode] = kernel.value();
        return;
    }
    if (mode == 4) {
        // the index arithmetic of kernels/grid_gradient_columns.h for the slabs by which the fused network sorts for this grid
        kernel::PointOrderKey key{};
        GradientColumnLayout layout;
        CHECK_ERROR(pointOrderKey(key, 0) && gradientColumns(key, layout), "this grid has no gradient columns");
        std::stringstream source;
        fillCode(source);
        source << "\n" << KernelLoader::MainFile("qmlp/kernels/grid_gradient_columns.h");
        const int flags = QuickMLP::Instance().getCompileFlags() | (compileOnly ? KernelLoader::CompileOnly : 0);
        auto kernel = QuickMLP::Instance().kernelLoader()->getKernel(
            "qmlp::kernel::GridGradientColumnsTraceKernel<" + layout.configType + ", " + std::to_string(layout.cellsPerSlab) + ">",
            source.str(), flags);
        if (!compileOnly) cornersKernel_[mode] = kernel.value();
        return;
    }
    {
        const std::string name = qualifiedName();
        const std::string source = standaloneSource(
            *this, "", "", name + "::corners(encodingInput, cEncoding, cornerIndices, cornerWeights);\n", "",
            name + "::traceGather(encodingInput, cEncoding, cornerIndices, cornerWeights);\n",
            name + "::traceScatter(lane, tileBase, numel, inputs, cEncoding, indices, weights);\n");
        const char* kernels[] = {"qmlp::kernel::EncodingCornersKernel", "qmlp::kernel::EncodingTraceKernel<1>",
                                 "qmlp::kernel::EncodingTraceKernel<2>"};
        const int flags = QuickMLP::Instance().getCompileFlags() | (compileOnly ? KernelLoader::CompileOnly : 0);
        auto kernel = QuickMLP::Instance().kernelLoader()->getKernel(kernels[mode], source, flags);
        if (!compileOnly) cornersKernel_[mode] = kernel.value();
    }
}

EncodingFactory::EncodingFactory()
{
    encodings_[EncodingIdentity::ID()] = [](const json& cfg) { return std::make_shared<EncodingIdentity>(cfg); };
    encodings_[EncodingHashGrid::ID()] = [](const json& cfg) { return std::make_shared<EncodingHashGrid>(cfg); };
    encodings_[EncodingLineIntegration::ID()] = [](const json& cfg) { return std::make_shared<EncodingLineIntegration>(cfg); };
}

EncodingFactory& EncodingFactory::Instance()
{
    static EncodingFactory INSTANCE;
    return INSTANCE;
}

static std::string lowerCase(std::string s)
{
    for (auto& c : s) c = static_cast<char>(std::tolower(static_cast<unsigned char>(c)));
    return s;
}

IEncoding_ptr EncodingFactory::create(const json& cfg)
{
    const std::string id = cfg.at("id").get<std::string>();
    auto it = encodings_.find(id);
    if (it == encodings_.end()) {
        // The reference matches the id exactly, but its own sample specifications write
        // "identity" for "Identity" (network_configs/test1.json:9, README.md:76): match
        // without regard to case.
        for (auto jt = encodings_.begin(); jt != encodings_.end(); ++jt)
            if (lowerCase(jt->first) == lowerCase(id)) it = jt;
    }
    if (it == encodings_.end()) throw configuration_error("No encoding with id '%s' found", id.c_str());
    return it->second(cfg);
}

QUICKMLP_NAMESPACE_END
