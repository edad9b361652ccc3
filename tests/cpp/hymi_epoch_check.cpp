// Host-only: every setting that changes what a captured cycle would launch, or frees a table that it reads, counts the
// mesh's schedule epoch up (a graph of an older epoch is captured again before it is replayed).
#include <cstdio>

#include "internal.hpp"

using namespace hymi;

static int failures = 0;
static void expectNew( const char* what, int level, uint64_t before, uint64_t after )
{
   if ( after == before )
   {
      std::printf( "%s on level %d left the epoch at %llu\n", what, level, (unsigned long long) after );
      failures++;
   }
}

int main()
{
   Context ctx;
   ctx.hostOnly = true;
   Mesh M;
   M.ctx             = &ctx;
   const double lo[] = { 0, 0, 0 }, hi[] = { 1, 1, 1 };
   M.T               = Topology::cuboid( lo, hi, 1, 1, 1 );
   for ( int level : { 4, 5, 6 } )
   {
      uint64_t      e = M.scheduleEpoch;
      MarchSchedule S;
      S.kind = 3, S.rows = 16, S.waves = 2, S.block = 1;
      M.setSchedule( level, S );
      expectNew( "setSchedule", level, e, M.scheduleEpoch );
      e = M.scheduleEpoch;
      M.setSchedule( level, S ); // the same again: its table is kept or rebuilt, a captured graph may not be replayed
      expectNew( "setSchedule again", level, e, M.scheduleEpoch );
      e = M.scheduleEpoch;
      M.setCellSor( level, 24, 3 );
      expectNew( "setCellSor 24", level, e, M.scheduleEpoch );
      e = M.scheduleEpoch;
      M.setCellSor( level, 0, 0 );
      expectNew( "setCellSor 0", level, e, M.scheduleEpoch );
      e = M.scheduleEpoch;
      M.setResidualRestrict( level, 1 );
      expectNew( "setResidualRestrict 1", level, e, M.scheduleEpoch );
      e = M.scheduleEpoch;
      M.setResidualRestrict( level, 0 );
      expectNew( "setResidualRestrict 0", level, e, M.scheduleEpoch );
   }
   std::printf( "%d failures\n", failures );
   return failures;
}
