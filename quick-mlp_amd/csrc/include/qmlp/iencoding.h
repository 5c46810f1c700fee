#pragma once

#include "common.h"
#include "json.h"
#include "kernel_loader.h"
#include "tensor.h"
#include <qmlp/kernels/encoding_level_shares.h>
#include <qmlp/kernels/grid_gradient_items.h>
#include <qmlp/kernels/point_order_key.h>

#include <functional>
#include <mutex>
#include <optional>
#include <sstream>
#include <unordered_map>
#include <vector>

QUICKMLP_NAMESPACE_BEGIN

/**
 * Defines an input encoding.
 *
 * What the device-side implementation must provide:
 * <code>
 * struct NameOfEncoding
 * {
 *     static constexpr int NumOutputs;
 *     template<typename I, typename O>
 *     static __device__ void forward(const I& input, O& output [, const param-type& params ]);
 *
 *     template<bool EvaluateInputGradients, bool EvaluateParameterGradients, typename I, typename O, typename AdjI>
 *     static __device__ void adjoint(const I& input, const O& adjOutput, AdjI& adjInput [, const param-type& params ]);
 * }
 * </code>
 * 'input' is indexable with operator[] and yields the raw float inputs of one point;
 * 'output' is indexable, assignable and has a typedef ValueType (float or a half type).
 * Encodings with parameters receive them as one by-value kernel argument of the type
 * named by parameterName(), whose bytes fillParameterMemory() produces.
 */
class IEncoding
{
public:
    virtual ~IEncoding() = default;

    [[nodiscard]] virtual json toJson() const = 0;
    [[nodiscard]] virtual std::string id() const = 0;

    /** The maximal addressed input channel, e.g. 2 for a 3D index. */
    [[nodiscard]] virtual int maxInputChannel() const = 0;

    /** The number of output channels */
    [[nodiscard]] virtual int numOutputChannels() const = 0;

    /** The qualified device type of the encoding including all template arguments. */
    [[nodiscard]] virtual std::string qualifiedName() const = 0;

    /** Appends the device code needed by qualifiedName(): includes and generated definitions. */
    virtual void fillCode(std::stringstream& code) const = 0;

    /** True iff the encoding has a parameter structure (and trainable parameters). */
    [[nodiscard]] virtual bool hasParameters() const { return false; }

    /** Fully-qualified device type of the parameter structure. */
    [[nodiscard]] virtual std::string parameterName() const { return ""; }

    [[nodiscard]] virtual Tensor::Precision parameterPrecision(Tensor::Usage usage) const { return Tensor::FLOAT; }

    [[nodiscard]] virtual int parameterCount() const { return 0; }

    /**
     * Sets the underlying parameter to the specified tensor: 1D with parameterCount()
     * entries of type parameterPrecision(usage). An undefined tensor clears it.
     */
    virtual void setParameter(const Tensor& tensor, Tensor::Usage usage) {}

    /** True iff a tensor is currently bound for this usage (always true without parameters). */
    [[nodiscard]] virtual bool hasParameterTensor(Tensor::Usage usage) const { return true; }

    /**
     * Writes the bytes of the parameter structure (kernel argument) into 'dst' with a
     * capacity of 'dstSize' bytes; returns the number of bytes written.
     */
    [[nodiscard]] virtual int fillParameterMemory(char* dst, int dstSize) { return 0; }

    /** Zeros the gradients of this encoding's parameters (no-op without parameters). */
    virtual void zeroGradients() {}

    /**
     * For the fused backward kernel: how many leading levels (or other leading parts) of the
     * parameter gradients a workgroup may sum in LDS before adding them to the gradient
     * tensor, if it has maxBytes of LDS for that. Returns the number of floats needed (0: none)
     * and sets 'levels', which the device code receives as scatterTile<levels>.
     */
    /**
     * Number of parameter tables that the fused forward kernel sweeps one after the other
     * (the levels of a grid). With two or more, the workgroups of a launch should stay in
     * step so that only the table in use occupies the L2; 0 for encodings without tables.
     */
    [[nodiscard]] virtual int numSweptTables() const { return 0; }

    /**
     * 32-bit registers that the gathers of one point from one table occupy while they are in
     * flight (all corners of a cell); 0 for encodings that gather nothing. The fused forward
     * kernel keeps the gathers of several points per lane in flight and sizes that number by it.
     */
    [[nodiscard]] virtual int gatherRegistersPerPoint() const { return 0; }

    /**
     * Encodings that gather from a table too large for the L2 of one accelerator die, and whose
     * gathers are close in memory for points that are close in space (dense grids), fill in how
     * points are assigned to slabs of that table and return true: the fused inference kernel
     * then evaluates the points slab by slab.
     * \param numPoints size of the batch; >0: only say yes if so many points are also expected
     *   to gain more from the order than the sort costs. 0: say whether an order exists at all.
     */
    [[nodiscard]] virtual bool pointOrderKey(kernel::PointOrderKey& key, long long numPoints = 0) const
    {
        (void)key;
        (void)numPoints;
        return false;
    }

    /** Output channels that the device code writes together (the features of a grid entry). */
    [[nodiscard]] virtual int channelsWrittenTogether() const { return 1; }

    /** Workgroups of the standalone forward kernel that may share out the levels of a point (device function forwardGroup; 1: forward). */
    [[nodiscard]] virtual int levelGroups() const { return 1; }

    /** Tiles of each level that a wavefront of EncodingLevelsKernel takes; empty: no such kernel. */
    [[nodiscard]] virtual std::vector<int> levelTiles() const { return {}; }

    /** Grids of many levels whose tile-wide adjoint the wavefronts of a workgroup may share by levels (device function
     *  adjointShared, for as many features as scatterTile() takes); 0 or the number of wavefronts. */
    [[nodiscard]] int sharedAdjointWaves() const
    {
        const int features = channelsWrittenTogether(), levels = numSweptTables();
        if (!hasParameters() || levelGroups() <= 1 || levels < 4 || (features & (features - 1)) != 0 || features > 32) return 0;
        return levels >= 8 ? 8 : 4;
    }
    static constexpr int SHARED_ADJOINT_MAX_BATCH = 256 * 64;   // a workgroup per compute unit

    /** One work item of GridGradientSlicesKernel (mirrors kernel::GridGradientSlice). */
    struct GradientSlice
    {
        int level;
        unsigned first;
        int floats;
        int slice;
        int part;
        int parts;
        int place;
        int slices;
    };
    /** The temporary memory of the kernels of kernels/grid_gradient.h (mirrors kernel::GridGradientWorkspace). */
    struct GradientWorkspace
    {
        void *records, *places, *exceptions, *largest;
        int regions, recordsPerRegion, largestCount, reserved;
    };
    /** What the host needs to run the kernels of kernels/grid_gradient.h for an encoding. */
    struct GradientSliceLayout
    {
        std::string configType;            // device type of the level table
        int sliceFloats = 0;               // floats of a full slice
        int recordWords = 0;               // 32-bit words of a record
        int pairs = 0;                     // records per point and level
        int features = 0;                  // floats of an entry
        int inputChannels = 0;             // coordinates of a point
        int pointsPerWorkgroup = 0;        // most lanes of a workgroup of the records kernel (a power of two)
        int derivativeBytesPerPoint = 0;   // of kernel::PositionDerivativeLayout: what a training pass may keep for the input gradients
        /** Dynamic LDS of the records kernel with this many lanes: its records of one level, and per slice of the level (at
         *  most 512) their number, that of the next level and the place of the first. */
        int recordsLdsBytes(int points) const { return points * pairs * recordWords * 4 + 3 * (512 + 1) * 4 + 64; }
        /** Dynamic LDS of the slice kernel: 64-bit sums of a slice and of the entry behind it. */
        int slicesLdsBytes() const { return (sliceFloats + features) * 8; }
        std::vector<int> slicesPerLevel;
        std::vector<GradientSlice> items;  // one workgroup of the slice kernel each
        int numSlices() const
        {
            int n = 0;
            for (int s : slicesPerLevel) n += s;
            return n;
        }
        /** Where the records kernel gets the gradients with respect to the input from: nowhere, the entries of all corners, or what the forward pass kept. */
        enum InputGradients { NO_INPUT_GRADIENTS = 0, FROM_ENTRIES = 1, FROM_DERIVATIVES = 2 };
        /** Workgroups of the records kernel over which the levels of a region are shared out, and all that work on a region (as GridGradientRecords::inputGradientsInline). */
        int levelGroups(InputGradients input) const { return input == FROM_ENTRIES ? 1 : std::min(8, static_cast<int>(slicesPerLevel.size())); }
        int workgroupsPerRegion(InputGradients input) const
        {
            const bool oneLevel = slicesPerLevel.size() == 1;
            const bool inputsApart = input == FROM_ENTRIES ? oneLevel : input == FROM_DERIVATIVES && !(oneLevel && pairs * recordWords > 16);
            return levelGroups(input) + (inputsApart ? 1 : 0);
        }
        /**
         * Regions that the records kernel works on at a time (of a large batch every workgroup gets several): a multiple of the dies,
         * so that the groups of a region run on the same one (see GridGradientRecordsKernel).
         */
        static int regionSlots(long long numel, int points)
        {
            constexpr int DIES = 8;
            return static_cast<int>(roundUp(std::min<long long>(divUp<long long>(numel, points), 1024), static_cast<long long>(DIES)));
        }
        /**
         * Lanes of a workgroup of GridGradientExceptionsKernel, and workgroups: as many as there are parts of lists, at most what the
         * chip holds, an odd number: lists have a power of two of parts, of which often only the first ones hold anything.
         */
        static constexpr int EXCEPTIONS_BLOCK = kernel::GRID_GRADIENT_EXCEPTIONS_BLOCK;
        int exceptionsGrid(const GradientWorkspace& workspace) const
        {
            return static_cast<int>(std::min<long long>(static_cast<long long>(workspace.regions) * static_cast<long long>(slicesPerLevel.size())
                                                            * divUp(workspace.recordsPerRegion, EXCEPTIONS_BLOCK), 1023));
        }
        /** The parts of the temporary memory for regions of so many points, and its bytes. */
        GradientWorkspace workspace(void* memory, long long numel, int points, InputGradients input, size_t* bytes = nullptr) const
        {
            GradientWorkspace w{};
            size_t offset = 0;
            auto take = [&](size_t size) {
                void* p = memory ? static_cast<char*>(memory) + offset : nullptr;
                offset += roundUp(size, size_t(256));
                return p;
            };
            w.regions = static_cast<int>(divUp<long long>(numel, points));
            w.recordsPerRegion = points * pairs;
            w.largestCount = regionSlots(numel, points) * levelGroups(input);
            const size_t levels = slicesPerLevel.size(), records = static_cast<size_t>(w.regions) * w.recordsPerRegion * levels;
            w.largest = take(static_cast<size_t>(w.largestCount) * sizeof(uint32_t));
            w.places = take(static_cast<size_t>(w.regions) * (numSlices() + 2 * levels) * sizeof(uint16_t));
            w.records = take(records * recordWords * sizeof(uint32_t));
            w.exceptions = take(records * sizeof(uint16_t));
            if (bytes) *bytes = offset;
            return w;
        }
        /** Bytes of temporary memory of a batch, whatever the size of its regions and the number of its groups. */
        size_t workspaceBytes(long long numel) const
        {
            size_t most = 0;
            for (int points = pointsPerWorkgroup; points >= std::min(128, pointsPerWorkgroup); points /= 2) {
                size_t bytes = 0;
                (void)workspace(nullptr, numel, points, NO_INPUT_GRADIENTS, &bytes);   // (of most groups)
                most = std::max(most, bytes);
            }
            return most;
        }
    };
    /** What the host needs to run the kernels of kernels/grid_gradient_columns.h for an encoding. */
    struct GradientColumnLayout
    {
        std::string configType;      // device type of the level table
        int cellsPerSlab = 0;        // cells per slab and sorted coordinate (the kernels' CPS)
        int owners = 0;              // owners per sorted coordinate: workgroups that share out the nodes of the grid
        int ldsBytes = 0;            // 64-bit sums of one owner
    };
    /**
     * Encodings whose parameter gradients, for a batch that is sorted by the slabs of `key` (pointOrderKey()), can
     * be summed owner by owner in LDS without any records (see kernels/grid_gradient_columns.h) return true and
     * fill in the layout.
     */
    [[nodiscard]] virtual bool gradientColumns(const kernel::PointOrderKey& key, GradientColumnLayout& layout) const
    {
        (void)key;
        (void)layout;
        return false;
    }

    /**
     * Encodings whose parameter gradients can be summed slice by slice in LDS instead of being
     * scattered with global atomics (see kernels/grid_gradient.h) return true and fill in the layout.
     * \param floatAdjoints the adjoint of the encoded rows is given in floats (standalone), else in halves (fused)
     */
    [[nodiscard]] virtual bool gradientSlices(GradientSliceLayout& layout, bool floatAdjoints = false) const
    {
        (void)layout;
        (void)floatAdjoints;
        return false;
    }

    /** gradientSlices(), worked out once (asked on every call): nullptr where there are none. */
    [[nodiscard]] const GradientSliceLayout* sliceLayout(bool floatAdjoints = false) const
    {
        const int k = floatAdjoints ? 1 : 0;
        std::call_once(sliceLayoutOnce_[k], [this, k] {
            GradientSliceLayout layout;
            if (gradientSlices(layout, k == 1)) sliceLayout_[k] = std::move(layout);
        });
        return sliceLayout_[k].has_value() ? &sliceLayout_[k].value() : nullptr;
    }

    /**
     * Whether the parameter gradients of a batch go through the slice kernels rather than through float atomics.
     * Below these sizes the two slice kernels cost more than the atomics they save (their work items zero and write
     * back whole slices whatever the batch). A train step of one dense 4-D level with 8 features at 2^14 / 2^15 / 2^16 /
     * 2^17 points 0.08 / 0.09 / 0.12 / 0.19 ms with atomics, 0.10 / 0.11 / 0.12 / 0.23 ms by slices. The atomics of a
     * point grow with the number of levels, the fixed work of the slice kernels with the size of the table: a train
     * step of a network behind a 16-level hash grid of halves at 2^12 / 2^13 / 2^14 / 2^15 points 71 / 86 / 119 / 192 us with
     * atomics, 84 / 76 / 90 / 103 us by slices (with input gradients 99 / 103 / 139 / 234 and 98 / 99 / 97 / 110 us, of which
     * the host's path is 90: no reason to go below 2^14); the adjoint pass of that grid alone, of floats, at 2^13 / 2^14 / 2^15 / 2^16
     * points 31 / 60 / 117 / 229 us with atomics and - / 46 / 51 / 61 by slices, with input gradients 43 / 76 / 157 / 279 and
     * - / 75 / 88 / 118 us.
     * \param manyLevelsMinBatch from which size on grids of 8 levels or more take the slices
     */
    static constexpr int SLICE_GRADIENTS_MIN_BATCH = 1 << 16;
    static constexpr int SLICE_GRADIENTS_MIN_BATCH_STANDALONE = 1 << 14, SLICE_GRADIENTS_MIN_BATCH_STANDALONE_INPUT = (1 << 14) + 1;
    static constexpr int SLICE_GRADIENTS_MIN_BATCH_TRAIN_STEP = 1 << 13, SLICE_GRADIENTS_MIN_BATCH_TRAIN_STEP_INPUT = 1 << 14;
    // (a pass without weight gradients needs no temporary memory for batches below)
    static constexpr int SLICE_GRADIENTS_MIN_BATCH_NO_WEIGHTS = 1 << 15;
    [[nodiscard]] static bool slicesPay(const GradientSliceLayout& layout, long long numel, int manyLevelsMinBatch)
    {
        return numel >= SLICE_GRADIENTS_MIN_BATCH || (numel >= manyLevelsMinBatch && layout.slicesPerLevel.size() >= 8);
    }

    [[nodiscard]] virtual int ldsGradientFloats(int maxBytes, int& levels) const
    {
        levels = 0;
        return 0;
    }

    /**
     * Standalone forward pass.
     * \param input shape (B, Cin), float32
     * \param output shape (B, >= numOutputChannels()), float32, unit stride along the channels
     * \param parametersForward optional override of the inference parameters for this call
     */
    virtual void forward(const Tensor& input, Tensor& output, stream_t stream,
                         const std::optional<const Tensor>& parametersForward);

    enum AdjointMode
    {
        INPUT_GRADIENTS = 0x1,
        PARAM_GRADIENTS = 0x2,
        ALL_GRADIENTS = INPUT_GRADIENTS | PARAM_GRADIENTS
    };

    /** Bytes of temporary device memory with which adjoint() is fastest for such a batch (0: it needs none). */
    [[nodiscard]] size_t adjointMemory(long long numel, int adjointMode) const;

    /**
     * Standalone adjoint pass; adjInput (B, Cin) and the parameter gradients are accumulated.
     */
    virtual void adjoint(const Tensor& input, const Tensor& adjOutput, Tensor& adjInput, stream_t stream,
                         const std::optional<const Tensor>& parametersForward,
                         const std::optional<const Tensor>& parametersGradients,
                         int adjointMode = AdjointMode::ALL_GRADIENTS);
    /**
     * \param tmpMemory adjointMemory() bytes at a multiple of 256, which belong to this call until its kernels have
     *    run; without them the parameter gradients are scattered with atomics
     * \param overwriteParameters with tmpMemory, where adjointMemory() is not 0: the parameter gradients are written
     *    instead of added to
     */
    void adjoint(const Tensor& input, const Tensor& adjOutput, Tensor& adjInput, stream_t stream,
                 const std::optional<const Tensor>& parametersForward,
                 const std::optional<const Tensor>& parametersGradients, int adjointMode, void* tmpMemory, bool overwriteParameters = false);

    /**
     * Compiles the standalone forward kernel and, for adjointMode > 0, the adjoint kernels of
     * that mode into the kernel cache without loading them; needs no GPU.
     */
    void precompile(int adjointMode = AdjointMode::ALL_GRADIENTS);

    /** The kernel that forward() takes for these tensors (diagnostics and tests; needs a device). */
    [[nodiscard]] std::string forwardKernelName(const Tensor& input, const Tensor& output) const;

private:
    std::string forwardKernelSource(int groups) const;
    std::string adjointKernelSource(int adjointMode, bool sharedTile = false) const;
    std::optional<KernelFunction> adjointSharedKernel_[AdjointMode::ALL_GRADIENTS + 1];
    std::optional<KernelFunction> forwardKernel_[2];   // [1]: by groups of levels
    /** Whether forward() takes EncodingLevelsKernel. */
    bool forwardByLevels(const Tensor& input, const Tensor& output) const;
    std::vector<KernelFunction> compileForwardByLevels(int flags) const;
    std::vector<KernelFunction> forwardByLevels_;      // EncodingLevelsKernel, EncodingRowsKernel
    // Where the kernel without groups is the faster one, see EncodingForwardKernel.
    static constexpr long long FORWARD_WHOLE_ROWS_MIN_BATCH = 3 << 14;
    std::optional<KernelFunction> adjointKernel_[AdjointMode::ALL_GRADIENTS + 1];
    mutable std::once_flag sliceLayoutOnce_[2];
    mutable std::optional<GradientSliceLayout> sliceLayout_[2];

    /** The kernels of kernels/grid_gradient.h for adjoints given in floats. */
    struct SliceKernels
    {
        // GridGradientRecordsKernel without / with input gradients, with pointsPerWorkgroup >> i lanes per workgroup
        std::vector<std::optional<KernelFunction>> records[2];
        std::optional<KernelFunction> slices, exceptions;
        Tensor items;
    };
    SliceKernels sliceKernels_;
    static int recordsVariants(const GradientSliceLayout& layout);
    std::optional<KernelFunction> compileRecords(const GradientSliceLayout& layout, bool inputGradients, int variant, int flags) const;
    /** GridGradientSlicesKernel and GridGradientExceptionsKernel */
    std::vector<KernelFunction> compileSlices(const GradientSliceLayout& layout, int flags) const;
    void adjointBySlices(const GradientSliceLayout& layout, const Tensor& input, const Tensor& adjOutput, Tensor& adjInput, stream_t stream,
                         int adjointMode, void* tmpMemory, char* parameters, bool overwriteParameters);
};
typedef std::shared_ptr<IEncoding> IEncoding_ptr;

/**
 * Encodings over a bounded volume; can serve as child of other encodings.
 */
class IVolumetricEncoding : public IEncoding
{
public:
    [[nodiscard]] virtual int ndim() const = 0;

    typedef std::vector<float> BoundingBoxVector_t;
    [[nodiscard]] virtual BoundingBoxVector_t boundingBoxMin() const = 0;
    [[nodiscard]] virtual BoundingBoxVector_t boundingBoxSize() const = 0;
    [[nodiscard]] virtual BoundingBoxVector_t boundingBoxInvSize() const = 0;
};

class EncodingFactory
{
private:
    EncodingFactory();
    typedef std::function<IEncoding_ptr(const json&)> factory_t;
    std::unordered_map<std::string, factory_t> encodings_;

public:
    static EncodingFactory& Instance();
    IEncoding_ptr create(const json& cfg);
};

QUICKMLP_NAMESPACE_END
