"""Generates imau_vel_bindings.f90 (ISO_C_BINDING mirror of include/imau_vel.h).

Run:  python imau-ice_amd/fortran/gen_bindings.py   (--stdout: print instead of writing)
The derived types are BIND(C), so the Fortran compiler lays them out like the
companion C compiler lays out the structs of the header.
"""
import os
import re
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.dirname(HERE))
from imau_vel import abi  # noqa: E402

FT = {"c_double": "REAL(C_DOUBLE)", "c_int": "INTEGER(C_INT32_T)", "c_long": "INTEGER(C_INT64_T)"}


def ftype(t):
    import ctypes
    if hasattr(t, "contents"):
        return "TYPE(C_PTR)", None
    if hasattr(t, "_length_"):
        return ftype(t._type_)[0], t._length_
    return {ctypes.c_double: "REAL(C_DOUBLE)", ctypes.c_int32: "INTEGER(C_INT32_T)",
            ctypes.c_int64: "INTEGER(C_INT64_T)"}[t], None


def typedef(name, cls):
    out = ["  TYPE, BIND(C) :: %s" % name]
    for fname, t in cls._fields_:
        ty, n = ftype(t)
        out.append("    %-20s :: %s%s" % (ty, fname, "(%d)" % n if n else ""))
    out.append("  END TYPE %s" % name)
    return "\n".join(out)


def main():
    consts = ["  INTEGER(C_INT32_T), PARAMETER :: %s = %d" % (k, v) for k, v in sorted(abi.ENUMS.items())]
    consts.append("  INTEGER(C_INT32_T), PARAMETER :: IMAU_NZ_MAX = %d" % abi.NZ_MAX)
    body = r"""! imau_vel_bindings.f90 -- GENERATED by gen_bindings.py from include/imau_vel.h; do not edit.
!
! ISO_C_BINDING interface to libimauvel.so for a Fortran host (IMAU-ICE's
! ice_velocity_module calls these; see ice_velocity_module_gpu.f90).
MODULE imau_vel_bindings
  USE ISO_C_BINDING
  IMPLICIT NONE

%s

%s

%s

%s

%s

  INTERFACE
    FUNCTION imau_vel_init(grid, cfg, ctx) BIND(C, name='imau_vel_init') RESULT(rc)
      IMPORT :: C_INT, C_PTR, imau_grid, imau_cfg
      TYPE(imau_grid), INTENT(IN) :: grid
      TYPE(imau_cfg),  INTENT(IN) :: cfg
      TYPE(C_PTR),     INTENT(OUT) :: ctx
      INTEGER(C_INT) :: rc
    END FUNCTION
    FUNCTION imau_vel_solve_diva(ctx, grid, cfg, io) BIND(C, name='imau_vel_solve_diva') RESULT(rc)
      IMPORT :: C_INT, C_PTR, imau_grid, imau_cfg, imau_ice_io
      TYPE(C_PTR), VALUE :: ctx
      TYPE(imau_grid),   INTENT(IN)    :: grid
      TYPE(imau_cfg),    INTENT(IN)    :: cfg
      TYPE(imau_ice_io), INTENT(INOUT) :: io
      INTEGER(C_INT) :: rc
    END FUNCTION
    FUNCTION imau_vel_solve_ssa(ctx, grid, cfg, io) BIND(C, name='imau_vel_solve_ssa') RESULT(rc)
      IMPORT :: C_INT, C_PTR, imau_grid, imau_cfg, imau_ice_io
      TYPE(C_PTR), VALUE :: ctx
      TYPE(imau_grid),   INTENT(IN)    :: grid
      TYPE(imau_cfg),    INTENT(IN)    :: cfg
      TYPE(imau_ice_io), INTENT(INOUT) :: io
      INTEGER(C_INT) :: rc
    END FUNCTION
    FUNCTION imau_vel_solve_sia(ctx, grid, cfg, io) BIND(C, name='imau_vel_solve_sia') RESULT(rc)
      IMPORT :: C_INT, C_PTR, imau_grid, imau_cfg, imau_ice_io
      TYPE(C_PTR), VALUE :: ctx
      TYPE(imau_grid),   INTENT(IN)    :: grid
      TYPE(imau_cfg),    INTENT(IN)    :: cfg
      TYPE(imau_ice_io), INTENT(INOUT) :: io
      INTEGER(C_INT) :: rc
    END FUNCTION
    SUBROUTINE imau_vel_finalize(ctx) BIND(C, name='imau_vel_finalize')
      IMPORT :: C_PTR
      TYPE(C_PTR), VALUE :: ctx
    END SUBROUTINE
    FUNCTION imau_vel_keep_memory(ctx, bytes, kept) BIND(C, name='imau_vel_keep_memory') RESULT(rc)
      IMPORT :: C_INT, C_INT64_T, C_PTR
      TYPE(C_PTR), VALUE :: ctx
      INTEGER(C_INT64_T), VALUE :: bytes
      INTEGER(C_INT64_T), INTENT(OUT) :: kept
      INTEGER(C_INT) :: rc
    END FUNCTION
    FUNCTION imau_vel_last_error(ctx) BIND(C, name='imau_vel_last_error') RESULT(msg)
      IMPORT :: C_PTR
      TYPE(C_PTR), VALUE :: ctx
      TYPE(C_PTR) :: msg
    END FUNCTION
    SUBROUTINE imau_vel_default_config(cfg) BIND(C, name='imau_vel_default_config')
      IMPORT :: imau_cfg
      TYPE(imau_cfg), INTENT(OUT) :: cfg
    END SUBROUTINE
    ! run_ice_dynamics_direct / _pc with update_ice_thickness (ref, geo: C_LOC or C_NULL_PTR)
    FUNCTION imau_run_ice_dynamics_direct(ctx, grid, cfg, tcfg, pcfg, scfg, io, ref, SMB_year, BMB, Hi_end, &
                                          geo, st, t_end) BIND(C, name='imau_run_ice_dynamics_direct') RESULT(rc)
      IMPORT :: C_INT, C_PTR, C_DOUBLE, imau_grid, imau_cfg, imau_thickness_cfg, imau_producer_cfg, &
                imau_timestep_cfg, imau_ice_io, imau_timestep_state
      TYPE(C_PTR), VALUE :: ctx
      TYPE(imau_grid),           INTENT(IN)    :: grid
      TYPE(imau_cfg),            INTENT(IN)    :: cfg
      TYPE(imau_thickness_cfg),  INTENT(IN)    :: tcfg
      TYPE(imau_producer_cfg),   INTENT(IN)    :: pcfg
      TYPE(imau_timestep_cfg),   INTENT(IN)    :: scfg
      TYPE(imau_ice_io),         INTENT(INOUT) :: io
      TYPE(C_PTR), VALUE :: ref
      REAL(C_DOUBLE),            INTENT(IN)    :: SMB_year(*), BMB(*)
      REAL(C_DOUBLE),            INTENT(OUT)   :: Hi_end(*)
      TYPE(C_PTR), VALUE :: geo
      TYPE(imau_timestep_state), INTENT(INOUT) :: st
      REAL(C_DOUBLE), VALUE :: t_end
      INTEGER(C_INT) :: rc
    END FUNCTION
    FUNCTION imau_run_ice_dynamics_pc(ctx, grid, cfg, tcfg, pcfg, scfg, io, ref, SMB_year, BMB, Hi_end, &
                                      geo, st, pc, t_end) BIND(C, name='imau_run_ice_dynamics_pc') RESULT(rc)
      IMPORT :: C_INT, C_PTR, C_DOUBLE, imau_grid, imau_cfg, imau_thickness_cfg, imau_producer_cfg, &
                imau_timestep_cfg, imau_ice_io, imau_timestep_state, imau_pc_state
      TYPE(C_PTR), VALUE :: ctx
      TYPE(imau_grid),           INTENT(IN)    :: grid
      TYPE(imau_cfg),            INTENT(IN)    :: cfg
      TYPE(imau_thickness_cfg),  INTENT(IN)    :: tcfg
      TYPE(imau_producer_cfg),   INTENT(IN)    :: pcfg
      TYPE(imau_timestep_cfg),   INTENT(IN)    :: scfg
      TYPE(imau_ice_io),         INTENT(INOUT) :: io
      TYPE(C_PTR), VALUE :: ref
      REAL(C_DOUBLE),            INTENT(IN)    :: SMB_year(*), BMB(*)
      REAL(C_DOUBLE),            INTENT(OUT)   :: Hi_end(*)
      TYPE(C_PTR), VALUE :: geo
      TYPE(imau_timestep_state), INTENT(INOUT) :: st
      TYPE(imau_pc_state),       INTENT(INOUT) :: pc
      REAL(C_DOUBLE), VALUE :: t_end
      INTEGER(C_INT) :: rc
    END FUNCTION
  END INTERFACE

CONTAINS

  ! copy the C error string of a context into a Fortran string
  FUNCTION imau_vel_error_text(ctx) RESULT(txt)
    TYPE(C_PTR), INTENT(IN) :: ctx
    CHARACTER(LEN=512) :: txt
    CHARACTER(KIND=C_CHAR), DIMENSION(:), POINTER :: p
    INTEGER :: k
    TYPE(C_PTR) :: cp
    INTERFACE
      FUNCTION strlen(s) BIND(C, name='strlen') RESULT(n)
        IMPORT :: C_PTR, C_SIZE_T
        TYPE(C_PTR), VALUE :: s
        INTEGER(C_SIZE_T) :: n
      END FUNCTION
    END INTERFACE
    txt = ' '
    cp = imau_vel_last_error(ctx)
    IF (.NOT. C_ASSOCIATED(cp)) RETURN
    CALL C_F_POINTER(cp, p, [INT(strlen(cp))])
    DO k = 1, MIN(SIZE(p), LEN(txt))
      txt(k:k) = p(k)
    END DO
  END FUNCTION imau_vel_error_text

END MODULE imau_vel_bindings
""" % ("\n".join(consts), typedef("imau_grid", abi.ImauGrid), typedef("imau_cfg", abi.ImauCfg),
       typedef("imau_ice_io", abi.ImauIceIO),
       "\n\n".join(typedef(n, c) for n, c in (
           ("imau_thickness_cfg", abi.ImauThicknessCfg), ("imau_producer_cfg", abi.ImauProducerCfg),
           ("imau_timestep_cfg", abi.ImauTimestepCfg), ("imau_refgeo_io", abi.ImauRefgeoIO),
           ("imau_producer_io", abi.ImauProducerIO), ("imau_timestep_state", abi.ImauTimestepState),
           ("imau_pc_state", abi.ImauPcState))))
    if "--stdout" in sys.argv:
        sys.stdout.write(body)
        return
    with open(os.path.join(HERE, "imau_vel_bindings.f90"), "w") as f:
        f.write(body)


if __name__ == "__main__":
    main()
