// Kernel code generator, emission of the fused chain kernel: phases, prefetch, item loops, LDS copy-out.
#include "hip_codegen_impl.hpp"
#include "hip_kernel.hpp"

namespace acro
{
namespace codegen
{

auto Generator::Emit(HipKernelPlan &plan) -> void
{
    const int K = static_cast<int>(subs.size());
    const int U = static_cast<int>(uvars.size());
    const std::string dimName = mk.GetDimensionedNameString();
    std::string variant = str(NB) + "/" + str(NT) + "/" + (opt.noalias ? "n" : "a") + (Positional() ? "p" : "u") +
                          "/" + str(envInt("ACRO_HIP_PERSIST")) + (envInt("ACRO_HIP_PIPELINE") > 0 ? "p" + str(envInt("ACRO_HIP_PIPELINE")) : "") +
                          (envInt("ACRO_HIP_WAVES_PER_EU") > 0 ? "w" + str(envInt("ACRO_HIP_WAVES_PER_EU")) : "");
    for (const auto &st : stores) variant += st.elide ? "e" : (st.inLds ? "l" : "g");
    for (int u = 0; u < U; ++u) variant += "s" + str(uvars[u].storage) + "@" + str(uvars[u].viewOffset);
    for (int g : opt.gathered) variant += "g" + str(g);
    char hex[32];
    std::snprintf(hex, sizeof(hex), "%016llx", static_cast<unsigned long long>(hashString(dimName + variant)));
    plan.module_name = std::string("acro_mk_") + hex;
    const std::string function_name = plan.module_name;

    std::ostringstream sched;
    sched << "batch index " << (batch >= 0 ? idxName[batch] : std::string("(none)")) << " extent " << E << ", " << NB
          << " per workgroup of " << NT << " lanes" << (entriesFastest ? ", numbered with the entry fastest" : "") << ", LDS " << ldsDoubles * 8 << " bytes\n";
    for (int k = 0; k < K; ++k)
    {
        const Sub &s = subs[k];
        sched << "  [" << k << "] " << s.text << " : lanes(";
        for (size_t j = 0; j < s.lane.size(); ++j) sched << (j ? "," : "") << idxName[s.lane[j]];
        sched << ")=" << s.laneCount << " tile(";
        for (size_t j = 0; j < s.tile.size(); ++j) sched << (j ? "," : "") << idxName[s.tile[j]];
        sched << ")=" << s.tileCount << " contraction=" << s.contrCount << (s.loopMode ? " looped" : " unrolled")
              << (s.fusedWithPrev ? " in-register after previous" : "") << " phase " << s.phase << "; operands:";
        for (size_t v = 0; v < s.in.size(); ++v)
        {
            static const char *const names[] = {"registers", "scalar", "lds", "global"};
            const Source src = SourceOf(k, static_cast<int>(v));
            sched << " " << uvars[s.in[v].uvar].name << "<-"
                  << (src == kFromGlobal && GatherSlot(s.in[v].uvar) >= 0 ? "gathered" : names[src]);
        }
        const UVarInfo &uo = uvars[s.out.uvar];
        const bool elided = !StoresToGlobal(k);
        sched << "; " << uo.name << "->" << (NeedsLdsCopy(k) ? "lds" : "")
              << (elided ? "" : (NeedsLdsCopy(k) ? "+global" : "global")) << "\n";
    }
    plan.schedule = sched.str();

    out << "// Generated by the acrotensor HIP code generator for gfx950.\n";
    {
        std::istringstream lines(plan.schedule);
        std::string l;
        while (std::getline(lines, l)) out << "// " << l << "\n";
    }
    out << "typedef const __attribute__((address_space(4))) double *acro_scalar_ptr;\n";
    for (int k = 0; k < K; ++k)
    {
        // two doubles in one load: only the 8-byte alignment that every operand has is promised
        if (SplitLanesTakePairs(k))
        {
            out << "typedef double acro_pair __attribute__((ext_vector_type(2), aligned(8)));\n";
            break;
        }
    }
    out << "\n";
    out << "extern \"C\" __global__ __launch_bounds__(" << NT << ") ";
    // experiment switch: ask the compiler for a register budget that lets this many wavefronts share a SIMD
    if (envInt("ACRO_HIP_WAVES_PER_EU") > 0)
        out << "__attribute__((amdgpu_waves_per_eu(" << envInt("ACRO_HIP_WAVES_PER_EU") << ", " << envInt("ACRO_HIP_WAVES_PER_EU") << "))) ";
    out << "void " << function_name << "(";
    out << ParamList();
    out << ")\n{\n";
    if (ldsDoubles > 0) out << "    __shared__ double lds[" << ldsDoubles << "];\n";
    std::set<int> scalarStores;
    for (int k = 0; k < K; ++k)
    {
        for (size_t v = 0; v < subs[k].in.size(); ++v)
        {
            if (SourceOf(k, static_cast<int>(v)) == kFromConstant)
                scalarStores.insert(uvars[subs[k].in[v].uvar].storage);
        }
    }
    for (int si : scalarStores)
        out << "    const acro_scalar_ptr C" << si << " = (acro_scalar_ptr)T" << si << ";\n";
    out << "    const int tid = threadIdx.x;\n";
    // Persistent form (ACRO_HIP_PERSIST=<workgroups per CU>): a fixed grid walks over the batch in a loop.
    const long totalGroups = (E + NB - 1) / NB;
    const long persist = envInt("ACRO_HIP_PERSIST");
    const long gridGroups = persist > 0 ? std::min<long>(totalGroups, persist * 256) : totalGroups;
    const bool looped = gridGroups < totalGroups;
    // Pipelined form of the persistent loop (ACRO_HIP_PIPELINE=1): the streaming inputs of every phase, the first
    // included, live in registers across iterations; a phase that has consumed its registers at once requests
    // the next batch entries' values, so that a workgroup never waits for device memory at the top of an
    // iteration and the memory system always holds requests of every resident workgroup.
    const bool pipelined = looped && envInt("ACRO_HIP_PIPELINE") > 0;
    const std::string loopHeader = "    for (int e0 = blockIdx.x * " + str(NB) + "; e0 < " + str(E) + "; e0 += " +
                                   str(gridGroups * NB) + ")\n    {\n";
    if (looped && !pipelined)
        out << loopHeader;
    else if (!looped && NumGatherSlots() > 0 && envInt("ACRO_HIP_XCD_RUN") >= 0 && totalGroups >= 2048)
    {
        // Operands read through an index map (a node vector under an element-to-node map): neighbouring workgroups
        // read the same lines of the source vector.  Hardware deals consecutive workgroup ids round-robin to the eight
        // XCDs, each with an L2 of its own, so every such line was fetched by two or three of them (p = 3 mass apply on
        // 64^3 elements: 140 MB of node-vector fetches for a vector of 57.5 MB).  Renumbered, each XCD gets runs of
        // neighbouring workgroups inside a block of 8 runs, and the device as a whole still moves through one window
        // (runs of 8 / 16 / 32 / 64 / 128 workgroups: 91.0 / 90.5 / 90.9 / 90.7 / 91.4 us against 93.9 us, tensors rotated).
        const long run = envInt("ACRO_HIP_XCD_RUN") > 0 ? envInt("ACRO_HIP_XCD_RUN") : 16;
        out << "    const unsigned b_ = blockIdx.x;\n";
        out << "    const unsigned g_ = b_ >= gridDim.x / " << 8 * run << "u * " << 8 * run << "u ? b_ : b_ / " << 8 * run << "u * " << 8 * run
            << "u + (b_ % 8u) * " << run << "u + (b_ / 8u) % " << run << "u;\n";
        out << "    const int e0 = (int)g_ * " << NB << ";\n    {\n";
    }
    else if (!looped)
        out << "    const int e0 = blockIdx.x * " << NB << ";\n    {\n";

    const bool guardBatch = (E % NB) != 0;

    bool anyStaged = false;
    for (size_t si = 0; si < stores.size(); ++si)
    {
        const Storage &st = stores[si];
        if (!st.staged || !st.inLds) continue;
        anyStaged = true;
        const UVarInfo &u = uvars[st.members[0]];
        out << "    {   // " << u.name << ": device memory -> LDS, once per workgroup\n";
        out << "        for (int i = tid; i < " << u.size << "; i += " << NT << ")\n        {\n";
        out << "            int r_ = i, a = " << st.ldsOffset << ";\n";
        long natural = u.size;
        for (size_t d = 0; d < st.dims.size(); ++d)
        {
            natural /= st.dims[d];
            if (d + 1 < st.dims.size())
                out << "            a += (r_ / " << natural << ") * " << st.ldsStride[d] << "; r_ %= " << natural << ";\n";
            else
                out << "            a += r_ * " << st.ldsStride[d] << ";\n";
        }
        out << "            lds[a] = T" << si << "[" << Lit(u.viewOffset) << " + i];\n        }\n    }\n";
    }
    if (anyStaged) out << "    __syncthreads();\n";

    // Work-item header: batch entry and lane indices of item `w` of the phase that kernel `ks` opens.
    auto emitHeader = [&](const Sub &s, const std::string &indent) {
        // A wavefront whose 64 items belong to one batch entry: say so, and the compiler turns loads that depend
        // on the entry alone into scalar loads.
        if (entriesFastest)
        {
            // entry fastest: a wavefront holds 64 consecutive entries of one row of lane indices
            out << indent << "const int b = w & " << NB - 1 << ";\n";
            out << indent << "const int e = e0 + b;\n";
            if (!s.lane.empty())
            {
                out << indent << "const int r_ = w / " << NB << ";\n";
                long st = s.laneCount;
                for (size_t j = 0; j < s.lane.size(); ++j)
                {
                    const int id = s.lane[j];
                    st /= extent[id];
                    out << indent << "const int " << IdxVar(id) << " = ";
                    if (j == 0)
                        out << "r_ / " << st << ";\n";
                    else
                        out << "(r_ / " << st << ") % " << extent[id] << ";\n";
                }
            }
            return;
        }
        if (s.laneCount % 64 == 0 && envInt("ACRO_HIP_WAVE_UNIFORM") >= 0)
            out << indent << "const int b = __builtin_amdgcn_readfirstlane(w / " << s.laneCount << ");\n";
        else
            out << indent << "const int b = w / " << s.laneCount << ";\n";
        out << indent << "const int e = e0 + b;\n";
        if (!s.lane.empty())
        {
            out << indent << "const int r_ = w - b * " << s.laneCount << ";\n";
            long st = s.laneCount;
            for (size_t j = 0; j < s.lane.size(); ++j)
            {
                const int id = s.lane[j];
                st /= extent[id];
                out << indent << "const int " << IdxVar(id) << " = ";
                if (j == 0)
                    out << "r_ / " << st << ";\n";
                else
                    out << "(r_ / " << st << ") % " << extent[id] << ";\n";
            }
        }
    };

    // Phases, the chains (a kernel plus the kernels applied in its registers) each of them runs side by side, and
    // what each may prefetch at kernel entry: the loads of streaming inputs of every phase after the first are
    // issued before the first phase starts, so that their latency overlaps with the earlier phases instead of
    // stalling a workgroup that few others can cover for.
    struct Chain
    {
        int first, last;
        long W;       // work items
        long offset;  // first item slot in the phase (multiple of the wavefront size)
        std::vector<std::vector<std::pair<std::string, std::string>>> loads;  // per kernel: prefetchable loads
        // per kernel and pass: memo key -> register name
        std::vector<std::vector<std::map<std::string, std::string>>> names;
    };
    struct Phase
    {
        std::vector<Chain> chains;
        long slots = 0, passes = 1;
        bool prefetched = false;
        bool carried = false;  // pipelined loop: the prefetched values are requested one iteration ahead
    };
    std::vector<Phase> phases;
    for (int k = 0; k < K;)
    {
        Chain c;
        c.first = k;
        c.last = k;
        while (c.last + 1 < K && subs[c.last + 1].fusedWithPrev) ++c.last;
        c.W = static_cast<long>(NB) * subs[k].laneCount;
        if (phases.empty() || subs[k].phase != subs[phases.back().chains.back().first].phase) phases.push_back(Phase());
        Phase &ph = phases.back();
        c.offset = ph.slots;
        ph.slots += (c.W + 63) / 64 * 64;
        ph.chains.push_back(c);
        k = c.last + 1;
    }
    for (auto &ph : phases)
    {
        if (ph.chains.size() == 1) ph.slots = ph.chains[0].W;
        ph.passes = (ph.slots + NT - 1) / NT;
    }

    long prefetchBudget = envInt("ACRO_HIP_PREFETCH") < 0 ? 0 : kPrefetchDoubles;
    // The first phase's own loads join the prefetch (ACRO_HIP_PREFETCH_FIRST=-1 switches that off): they are then
    // requested ahead of the later phases' inputs, and since a wavefront's loads complete in the order they were
    // issued, the first phase starts as soon as its own operands are there instead of after everything that was
    // prefetched (p=7 diffusion apply: 960 -> 943 us).  Only when some later phase prefetches at all.
    const bool firstToo = pipelined || envInt("ACRO_HIP_PREFETCH_FIRST") >= 0;
    // Several chains in the first phase that fill their wavefronts in part: their loads stand behind two branches each, and
    // run-time compilers before ROCm 7.2 then hold all that is prefetched through the phases in between (diffusion apply at
    // p = 4, 6^3 points 97 registers instead of 44, and so on), which costs more wavefronts than the order of the loads
    // gains: from five values per lane on they stay in their phase.  Inputs changing, 2^22 points, us, prefetched -> in the
    // phase: p = 4, 6^3 65.9 -> 59.0, p = 5, 6^3 / 7^3 81.2 -> 67.1 / 73.8 -> 61.0, p = 6, 7^3 / 8^3 78.3 -> 67.3 / 86.0 -> 63.3,
    // p = 8, 9^3 / 10^3 83.5 -> 75.2 / 114.7 -> 73.9; four values, p = 3, 4^3 / 5^3 62.3 / 63.6 and 59.2 / 60.6; whole
    // wavefronts, p = 7, 8^3 to 10^3, 1 to 3 % slower in the phase.  With 7.2: p = 4, 6^3 59.5 / 59.2, p = 6, 8^3 63.4 / 63.2,
    // p = 8, 9^3 / 10^3 74.0 / 75.0 and 71.7 / 73.2.
    bool firstInPart = phases[0].chains.size() > 1 && !pipelined && RunTimeCompilerVersion() < 702;
    {
        bool whole = true;
        for (const Chain &c : phases[0].chains) whole = whole && 10 * c.W >= 9 * ((c.W + 63) / 64 * 64);
        firstInPart = firstInPart && !whole;
    }
    // Later phases first (they have the latency to hide), the first phase last, with what is left of the budget.
    std::vector<size_t> phaseOrder;
    for (size_t pi = 1; pi < phases.size(); ++pi) phaseOrder.push_back(pi);
    if (firstToo && phases.size() > 1) phaseOrder.push_back(0);
    bool anyLater = false;
    long firstPrefetchDoubles = 0, laterPrefetchDoubles = 0;  // registers per lane
    for (size_t pi : phaseOrder)
    {
        // ... or on its own when its items take several passes of the workgroup: all passes request their operands
        // before the first one uses them, instead of one round trip to device memory per pass
        // (ACRO_HIP_PREFETCH_PASSES=-1 switches that off).
        // Groups of one phase keep their item loop: with everything requested up front they measured the same
        // within noise (24 streaming shapes, geometric mean 74.1 against 74.0 % of the HBM peak); the two-step
        // 27 x 27 element matrix times element vector gained, 52.8 -> 57.6 %.
        const bool severalPasses = phases[0].passes > 1 && phases.size() > 1 && envInt("ACRO_HIP_PREFETCH_PASSES") >= 0;
        if (pi == 0 && !anyLater && !pipelined && !severalPasses) break;
        Phase &ph = phases[pi];
        long perLane = 0;  // registers one lane needs: a lane serves at most one chain per pass
        bool ok = true;
        for (auto &c : ph.chains)
        {
            c.loads.assign(c.last - c.first + 1, {});
            ForwardMap forwarded;
            long perPass = 0;
            for (int kk = c.first; kk <= c.last; ++kk)
            {
                if (subs[kk].loopMode)
                {
                    ok = false;
                    break;
                }
                std::vector<std::string> scratchLines;
                EmitUnrolledBody(kk, forwarded, scratchLines, nullptr, &c.loads[kk - c.first]);
                perPass += static_cast<long>(c.loads[kk - c.first].size());
            }
            perLane = std::max(perLane, perPass);
        }
        if (!ok || perLane == 0 || perLane * ph.passes > prefetchBudget || (pi == 0 && firstInPart && perLane >= 5)) continue;
        prefetchBudget -= perLane * ph.passes;
        (pi == 0 ? firstPrefetchDoubles : laterPrefetchDoubles) += perLane * ph.passes;
        ph.prefetched = true;
        anyLater = anyLater || pi > 0;
        // ACRO_HIP_PIPELINE=<n>: phases that hold at most n doubles per lane are carried across iterations (the
        // first phase always is: its inputs are what an iteration would otherwise start by waiting for)
        ph.carried = pipelined && (pi == 0 || perLane * ph.passes <= envInt("ACRO_HIP_PIPELINE"));
    }

    // Emits, for pass j of a phase (or for the item loop when j < 0), the selection of the chain a lane works
    // for and calls `body` inside the guarded scope of one work item.
    // A streaming group (one phase, no LDS) over few batch entries would leave most of the device idle with one
    // workgroup per entry: the passes of its item loop become workgroups of a second grid dimension instead.
    const long splitY = (phases.size() == 1 && ldsDoubles == 0 && !looped && phases[0].passes > 1 && totalGroups < 2048)
                            ? std::min<long>(phases[0].passes, 65535)
                            : 1;
    auto emitItems = [&](const Phase &ph, long j, const std::function<void(const Chain &, const std::string &)> &body) {
        std::string indent = "        ";
        if (j < 0 && splitY > 1)
            out << "    for (int w0 = tid + blockIdx.y * " << NT << "; w0 < " << ph.slots << "; w0 += " << splitY * NT
                << ")\n    {\n";
        else if (j < 0)
            out << "    for (int w0 = tid; w0 < " << ph.slots << "; w0 += " << NT << ")\n    {\n";
        else
            out << "    {\n        const int w0 = tid + " << j * NT << ";\n";
        for (size_t ci = 0; ci < ph.chains.size(); ++ci)
        {
            const Chain &c = ph.chains[ci];
            const long end = c.offset + (ph.chains.size() == 1 ? c.W : (c.W + 63) / 64 * 64);
            if (ph.chains.size() > 1)
            {
                out << indent << (ci ? "else if" : "if") << " (w0 < " << end << ")\n" << indent << "{\n";
                indent += "    ";
            }
            out << indent << "const int w = w0 - " << c.offset << ";\n";
            out << indent << "if (w < " << c.W << ")\n" << indent << "{\n";
            emitHeader(subs[c.first], indent + "    ");
            std::string inner = indent + "    ";
            if (guardBatch)
            {
                out << inner << "if (e < " << E << ")\n" << inner << "{\n";
                inner += "    ";
            }
            body(c, inner);
            if (guardBatch) out << indent << "    }\n";
            out << indent << "}\n";
            if (ph.chains.size() > 1)
            {
                indent.resize(indent.size() - 4);
                out << indent << "}\n";
            }
        }
        out << "    }\n";
    };

    // Whether exact wait counts pay was measured.  They do when three or four workgroups share a compute unit (p=7
    // diffusion apply, 53 KB of LDS each: the early phases of a workgroup must not wait for its whole prefetch,
    // 941 -> 931 us) and when the prefetch is no bigger than twice what the first phase reads anyway (mass apply
    // at p = 6 - 8: 97 -> 94 us).  With five or more workgroups per unit and a prefetch many times the first phase's
    // operands (p=5 and p=6 diffusion apply) the others cover the wait, and workgroups that run their phases back to
    // back once everything has arrived were faster, 184 -> 175 us: the loads stay behind their branch there.
    // ACRO_HIP_PREFETCH_CLAMP=-1 / =1 force the choice.
    const long ldsBytesPerGroup = (std::max<long>(1, ldsDoubles) * 8 + 1279) / 1280 * 1280;
    const bool clampPrefetch =
        envInt("ACRO_HIP_PREFETCH_CLAMP") > 0 ||
        (envInt("ACRO_HIP_PREFETCH_CLAMP") == 0 &&
         (160 * 1024 / ldsBytesPerGroup <= 4 || laterPrefetchDoubles <= 2 * firstPrefetchDoubles));
    // Requests the prefetched inputs of one phase for the batch entries that start at the `e0` in scope.
    auto emitPrefetchLoads = [&](const Phase &ph) {
        for (long j = 0; j < ph.passes; ++j)
        {
            auto loadsOf = [&](const Chain &c, const std::string &indent) {
                for (int kk = c.first; kk <= c.last; ++kk)
                {
                    if (c.loads[kk - c.first].empty()) continue;
                    Body bases;
                    EmitBases(kk, bases);
                    for (const auto &l : bases.bases) out << indent << l << "\n";
                    for (const auto &ld : c.loads[kk - c.first])
                        out << indent << c.names[kk - c.first][j].at(ld.first) << " = " << ld.second << ";\n";
                }
            };
            // A phase of one chain: lanes past the last work item request the last item's operands instead of
            // nothing.  The requests then sit in straight-line code, and the compiler can count exactly how
            // many loads were issued after the ones an earlier phase waits for (behind a branch it has to assume
            // none, and that phase would wait for everything that was prefetched).
            if (ph.chains.size() == 1 && clampPrefetch)
            {
                const Chain &c = ph.chains[0];
                out << "    {\n        const int w0 = tid + " << j * NT << ";\n";
                if (guardBatch)
                {
                    // the last workgroup may hold fewer batch entries: its last item is that of its last entry
                    out << "        const int wlast = (" << E << " - e0 < " << NB << " ? " << E << " - e0 : " << NB << ") * "
                        << subs[c.first].laneCount << " - 1;\n";
                    out << "        const int w = w0 < wlast ? w0 : wlast;\n";
                }
                else
                    out << "        const int w = w0 < " << c.W << " ? w0 : " << c.W - 1 << ";\n";
                emitHeader(subs[c.first], "        ");
                loadsOf(c, "        ");
                out << "    }\n";
                continue;
            }
            emitItems(ph, j, loadsOf);
        }
    };
    for (auto &ph : phases)
    {
        if (!ph.prefetched) continue;
        out << "    // streaming inputs of phase " << subs[ph.chains[0].first].phase
            << (pipelined ? ", held in registers across iterations\n" : ", requested before the first phase\n");
        for (auto &c : ph.chains)
            c.names.assign(c.last - c.first + 1, std::vector<std::map<std::string, std::string>>(ph.passes));
        for (long j = 0; j < ph.passes; ++j)
        {
            // One register set per pass, shared by the chains (a lane serves one chain in a pass).
            long widest = 0;
            for (auto &c : ph.chains)
            {
                long n = 0;
                for (int kk = c.first; kk <= c.last; ++kk)
                {
                    for (const auto &ld : c.loads[kk - c.first])
                        c.names[kk - c.first][j][ld.first] = "pf" + str(subs[c.first].phase) + "_" + str(j) + "_" + str(n++);
                }
                widest = std::max(widest, n);
            }
            for (long n = 0; n < widest; ++n)
                out << "    double pf" << subs[ph.chains[0].first].phase << "_" << j << "_" << n << " = 0.0;\n";
        }
        if (!pipelined) emitPrefetchLoads(ph);
    }
    if (pipelined)
    {
        out << "    {   // the first batch entries of this workgroup\n    const int e0 = blockIdx.x * " << NB << ";\n";
        for (const auto &ph : phases)
        {
            if (ph.carried) emitPrefetchLoads(ph);
        }
        out << "    }\n" << loopHeader;
        for (const auto &ph : phases)
        {
            if (ph.prefetched && !ph.carried) emitPrefetchLoads(ph);  // requested at the top of every iteration
        }
    }

    // results of phase `previous` that leave through their LDS tiles (after the barrier that ends it)
    auto emitCopyOut = [&](int previous) {
            for (int k = 0; k < K; ++k)
            {
                if (subs[k].phase != previous || !CopiesOutFromLds(k)) continue;
                const Storage &st = StoreOf(subs[k].out.uvar);
                const bool streams = envInt("ACRO_HIP_NT_STORE") >= 0 && (static_cast<long>(ldsDoubles) * 8 <= 20 * 1024 || envInt("ACRO_HIP_NT_COPY_OUT") >= 0);
                out << "    {   // " << uvars[subs[k].out.uvar].name << ": LDS tiles -> device memory\n";
                if (guardBatch)
                    out << "        const int count = (" << E << " - e0 < " << NB << " ? " << E << " - e0 : " << NB << ") * "
                        << st.tileSize << ";\n";
                else
                    out << "        const int count = " << static_cast<long>(NB) * st.tileSize << ";\n";
                out << "        double *dst = " << PtrName(subs[k].out.uvar) << " + e0 * " << Lit(st.tileSize) << ";\n";
                out << "        for (int i = tid; i < count; i += " << NT << ") ";
                if (streams)
                    out << "__builtin_nontemporal_store(lds[" << st.ldsOffset << " + i], &dst[i]);\n";
                else
                    out << "dst[i] = lds[" << st.ldsOffset << " + i];\n";
                out << "    }\n";
            }
    };
    bool first = true;
    for (const Phase &ph : phases)
    {
        if (!first) out << "    __syncthreads();\n";
        if (!first) emitCopyOut(subs[ph.chains[0].first].phase - 1);
        first = false;
        const long npass = ph.prefetched ? ph.passes : 1;
        for (long j = 0; j < npass; ++j)
        {
            emitItems(ph, ph.prefetched ? j : -1, [&](const Chain &c, const std::string &indent) {
                ForwardMap forwarded;
                for (int kk = c.first; kk <= c.last; ++kk)
                {
                    std::vector<std::string> lines;
                    if (subs[kk].loopMode)
                        EmitLoopBody(kk, lines);
                    else
                        EmitUnrolledBody(kk, forwarded, lines, ph.prefetched ? &c.names[kk - c.first][j] : nullptr);
                    // Scopes nest (closed after the chain) so that a kernel applied in registers sees the
                    // values of its producer.
                    out << indent << "{\n";
                    for (const auto &l : lines) out << indent << "    " << l << "\n";
                }
                for (int kk = c.first; kk <= c.last; ++kk) out << indent << "}\n";
            });
        }
        if (ph.carried)
        {
            out << "    {   // the same inputs of this workgroup's next batch entries\n";
            out << "    const int e0_next = e0 + " << gridGroups * NB << ";\n    if (e0_next < " << E << ")\n    {\n";
            out << "    const int e0 = e0_next;\n";
            emitPrefetchLoads(ph);
            out << "    }\n    }\n";
        }
    }
    {
        bool lastCopies = false;
        for (int k = 0; k < K; ++k) lastCopies = lastCopies || (subs[k].phase == subs.back().phase && CopiesOutFromLds(k));
        if (lastCopies)
        {
            out << "    __syncthreads();\n";
            emitCopyOut(subs.back().phase);
        }
    }
    if (looped && ldsDoubles > 0) out << "    __syncthreads();\n";
    out << "    }\n}\n";

    plan.source = out.str();
    HipLaunch launch;
    launch.function_name = function_name;
    launch.grid = static_cast<unsigned>(gridGroups);
    launch.grid_y = static_cast<unsigned>(splitY);
    launch.block = static_cast<unsigned>(NT);
    for (int si = 0; si < NumParamStores(); ++si) launch.params.push_back(si);
    for (int g = 0; g < NumGatherSlots(); ++g)
    {
        launch.params.push_back(-2 - 2 * g);
        launch.params.push_back(-3 - 2 * g);
    }
    plan.gathers_applied = NumGatherSlots() > 0;
    plan.launches.push_back(launch);
    plan.nb = NB;
    plan.lds_bytes = ldsDoubles * 8;
    FillParams(plan, true);
    for (const auto &s : subs)
    {
        if (s.out.repeated && s.op == '=')
            plan.zero_fills.push_back({uvars[s.out.uvar].storage, uvars[s.out.uvar].viewOffset, s.out.size});
    }
}

}  // namespace codegen
}  // namespace acro
