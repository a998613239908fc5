// Which steps of a plan the executor puts into one launch, without a GPU: the
// launchers defined here take the place of the library's and only note what
// they are asked for.  Plans as a custom dispatcher may record them, whose steps
// do not each start at the level the one before ended with, and one whose steps do.
#include <stdio.h>

#include <vector>

#include "pyramid_internal.hpp"

namespace {
struct Launch
{
  char kind;  // F: a fast step, G: a general one, T: a tail
  uint32_t inputLevel, successor;
};
std::vector<Launch> gLaunches;
std::vector<NvproPyramidStep> gPlan;

uint32_t record(NvproPyramidCmd* cmd, const NvproPyramidState* state)
{
  for(const NvproPyramidStep& s : gPlan)
    if(nvproPyramidCmdDispatch(cmd, s.pipeline, s.inputLevel << NVPRO_PYRAMID_INPUT_LEVEL_SHIFT | s.levelCount, 1u))
      return 0u;
  return state->remainingLevels;
}
}  // namespace

namespace nvpro_pyramid {
hipError_t launchFast(hipStream_t, const ImageDesc&, uint32_t inputLevel, uint32_t, uint32_t, const NextStep* next,
                      const TailPlan*)
{
  gLaunches.push_back({'F', inputLevel, next ? next->kind : 0u});
  return hipSuccess;
}
hipError_t launchTail(hipStream_t, const ImageDesc&, const TailPlan& plan)
{
  gLaunches.push_back({'T', plan.steps[0].inputLevel, 0u});
  return hipSuccess;
}
// Every general step that would be launched alone goes through these.
uint32_t tileSteps(const ImageDesc&, const NvproPyramidStep* steps, uint32_t, uint32_t*, uint32_t*)
{
  return steps[0].pipeline == NVPRO_PYRAMID_PIPELINE_GENERAL ? 1u : 0u;
}
hipError_t launchTiles(hipStream_t, const ImageDesc&, const TailPlan& plan, uint32_t, uint32_t)
{
  gLaunches.push_back({'G', plan.steps[0].inputLevel, 0u});
  return hipSuccess;
}
}  // namespace nvpro_pyramid

using namespace nvpro_pyramid;

struct Step
{
  uint32_t pipeline, inputLevel, levelCount;
};
constexpr uint32_t F = NVPRO_PYRAMID_PIPELINE_FAST, G = NVPRO_PYRAMID_PIPELINE_GENERAL;

// Compares the launches of a plan over a side x side image with `want`.
static int check(const char* what, uint32_t side, const std::vector<Step>& plan, const std::vector<Launch>& want)
{
  gPlan.clear();
  for(const Step& s : plan)
    gPlan.push_back(NvproPyramidStep{s.pipeline, s.inputLevel, s.levelCount});
  static uint32_t texels[4];
  const NvproPyramidPipelines pipes{NVPRO_PYRAMID_FORMAT_SRGBA8, 1u, 0u, 0u};
  NvproPyramidImage image{};
  image.data  = texels;  // never accessed: no kernel runs
  image.width = image.height = side;
  ImageDesc desc;
  NvproPyramidStep steps[kMaxPlanSteps];
  uint32_t count = 0, launches = 0;
  if(prepareImage(&pipes, &image, 0u, record, record, &desc, steps, &count, "check"))
  {
    fprintf(stderr, "%s: %s\n", what, nvproPyramidGetLastError());
    return 1;
  }
  gLaunches.clear();
  static uint32_t arrive[1];
  if(executePlan(nullptr, desc, steps, count, arrive, &launches) != hipSuccess || launches != gLaunches.size())
  {
    fprintf(stderr, "%s: failed, %zu launches\n", what, gLaunches.size());
    return 1;
  }
  bool same = gLaunches.size() == want.size();
  for(size_t k = 0; same && k < want.size(); ++k)
    same = gLaunches[k].kind == want[k].kind && gLaunches[k].inputLevel == want[k].inputLevel
           && gLaunches[k].successor == want[k].successor;
  if(!same)
  {
    fprintf(stderr, "%s:", what);
    for(const Launch& l : gLaunches)
      fprintf(stderr, " %c%u+%u", l.kind, l.inputLevel, l.successor);
    fprintf(stderr, "\n");
  }
  return same ? 0 : 1;
}

int main()
{
  int wrong = 0;
  // A one-group fast successor that reads the middle level of the step before it.
  wrong += check("fast successor of a middle level", 128u, {{F, 0, 3}, {F, 1, 3}, {F, 4, 3}},
                 {{'F', 0, 0}, {'T', 1, 0}});
  // The rest of the plan goes back a level, at once and later on.
  wrong += check("step back behind a fast successor", 128u, {{F, 0, 3}, {F, 3, 1}, {F, 3, 2}, {F, 5, 2}},
                 {{'F', 0, kNextFast}, {'T', 3, 0}});
  wrong += check("step back in a tail", 128u, {{F, 0, 3}, {G, 3, 1}, {F, 3, 2}, {F, 5, 2}},
                 {{'F', 0, 0}, {'G', 3, 0}, {'T', 3, 0}});
  // A tail that does not start at the step's last level.
  wrong += check("tail of a middle level", 128u, {{F, 0, 4}, {G, 3, 2}, {G, 5, 2}}, {{'F', 0, 0}, {'T', 3, 0}});
  // Steps in order keep their one launch.
  wrong += check("fast successor", 4096u, {{F, 0, 6}, {F, 6, 6}}, {{'F', 0, kNextFast}});
  wrong += check("tail", 128u, {{F, 0, 3}, {G, 3, 2}, {G, 5, 2}}, {{'F', 0, kNextTail}});
  printf("%d plans wrong\n", wrong);
  return wrong ? 1 : 0;
}
